"""GPU parity tests of the grouped GEMM: against the CPU oracle at small sizes and against an
fp32 torch formulation on the GPU at the benchmark shapes.  Tolerance: relative Frobenius
error <= 1e-2 (bf16/f16 inputs, fp32 accumulation)."""
import ctypes
import math

import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

TOL = 1e-2


@pytest.fixture(scope='module')
def gg():
    from megablocks_amd import grouped_gemm_util as gg
    return gg


def rel_err(a, b):
    a, b = a.double(), b.double()
    return float((a - b).norm() / b.norm().clamp_min(1e-30))


def max_block_err(got, ref, bm=64, bn=128):
    """Largest relative error over bm x bn blocks of the last two dimensions: one wrong piece of one tile
    shows here even where the error over the whole output would hide it."""
    got, ref = got.double(), ref.double()
    r, c = ref.shape[-2:]
    pr, pc = (-r) % bm, (-c) % bn
    d = torch.nn.functional.pad(got - ref, (0, pc, 0, pr))
    b = torch.nn.functional.pad(ref, (0, pc, 0, pr))
    shape = d.shape[:-2] + ((r + pr) // bm, bm, (c + pc) // bn, bn)
    num = d.reshape(shape).pow(2).sum(dim=(-3, -1)).sqrt()
    den = b.reshape(shape).pow(2).sum(dim=(-3, -1)).sqrt()
    scale = ref.norm() / max(1, num.numel()) ** 0.5              # a typical block norm, for blocks that are almost zero
    return float((num / torch.maximum(den, scale * 0.1)).max())


def _sizes(groups, rows, seed, empty=()):
    g = torch.Generator().manual_seed(seed)
    cuts = torch.sort(torch.randint(0, rows + 1, (groups - 1,), generator=g))[0]
    sizes = torch.diff(torch.cat([torch.zeros(1, dtype=torch.int64), cuts, torch.tensor([rows])]))
    for e in empty:                      # force some empty groups, keep the total
        if e + 1 < groups:
            sizes[e + 1] += sizes[e]
            sizes[e] = 0
    return sizes


def _units():
    return torch.cuda.get_device_properties(0).multi_processor_count


def _ref_gpu(a, b, sizes, trans_a, trans_b):
    a, b = a.float(), b.float()
    outs, start = [], 0
    for e, n in enumerate(sizes.tolist()):
        ae = a[start:start + n]
        if trans_a:
            outs.append(ae.t() @ b[start:start + n])
        else:
            outs.append(ae @ (b[e].t() if trans_b else b[e]))
        start += n
    return torch.stack(outs) if trans_a else torch.cat(outs)


SMALL = [  # groups, rows, k, n
    (1, 128, 128, 128), (4, 512, 64, 256), (8, 1000, 256, 512), (3, 777, 72, 40), (5, 300, 100, 36),
    (2, 64, 8, 8), (16, 2048, 512, 1408), (4, 50, 33, 17), (1, 1, 16, 16), (8, 4096, 1024, 256),
]


@pytest.mark.parametrize('groups,k,n', [(1, 64, 256), (59, 1440, 704), (56, 960, 1104), (174, 1344, 256), (5, 33, 17)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float32])
@pytest.mark.parametrize('sizes_on_device', [False, True])
def test_gmm_with_no_rows_at_all(gg, groups, k, n, dtype, sizes_on_device):
    """Every expert empty: the weight gradients (trans_a) are exact zeros written over whatever the output
    buffer held, and the row products are empty."""
    sizes = torch.zeros(groups, dtype=torch.int64)
    bs = sizes.cuda() if sizes_on_device else sizes
    a = torch.empty(0, k, device='cuda', dtype=dtype)
    c = torch.full((groups, k, n), float('nan'), device='cuda', dtype=dtype)
    out = gg.backend.gmm(a, torch.empty(0, n, device='cuda', dtype=dtype), bs, trans_a=True, c=c)
    assert out.shape == (groups, k, n) and int(torch.count_nonzero(out)) == 0
    w = torch.randn(groups, k, n, device='cuda').to(dtype)
    assert gg.backend.gmm(a, w, bs).shape == (0, n)
    assert gg.backend.gmm(torch.empty(0, n, device='cuda', dtype=dtype), w, bs, trans_b=True).shape == (0, k)


@pytest.mark.parametrize('groups,rows,k,n', SMALL)
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize('mode', ['nn', 'nt', 'tn'])
def test_gmm_vs_oracle(gg, groups, rows, k, n, dtype, mode):
    sizes = _sizes(groups, rows, seed=groups * 1000 + rows, empty=(1,) if groups > 2 else ())
    a = torch.randn(rows, k).to(dtype)
    if mode == 'tn':
        b = torch.randn(rows, n).to(dtype)
    elif mode == 'nt':
        b = (torch.randn(groups, n, k) * 0.1).to(dtype)
    else:
        b = (torch.randn(groups, k, n) * 0.1).to(dtype)
    want = oracle.gmm(a, b, sizes, trans_a=mode == 'tn', trans_b=mode == 'nt')
    got = gg.backend.gmm(a.cuda(), b.cuda(), sizes, trans_a=mode == 'tn', trans_b=mode == 'nt')
    assert got.shape == want.shape and got.dtype == dtype
    assert rel_err(got.cpu(), want) < TOL
    if mode == 'tn':
        for e, s in enumerate(sizes.tolist()):
            if s == 0:
                assert torch.count_nonzero(got[e]) == 0          # unused expert: exactly zero gradient
    got_dev = gg.backend.gmm(a.cuda(), b.cuda(), sizes.cuda().int(), trans_a=mode == 'tn', trans_b=mode == 'nt')
    assert torch.equal(got_dev, got)                              # device-resident sizes: same kernel, same result


def test_gmm_c_argument_and_errors(gg):
    sizes = torch.tensor([100, 28])
    a = torch.randn(128, 64).bfloat16().cuda()
    b = torch.randn(2, 64, 32).bfloat16().cuda()
    c = torch.full((128, 32), 7.0).bfloat16().cuda()
    out = gg.backend.gmm(a, b, sizes, c=c)
    assert out is c and rel_err(c.cpu(), oracle.gmm(a.cpu(), b.cpu(), sizes)) < TOL
    with pytest.raises(ValueError):
        gg.backend.gmm(a, b, sizes, c=torch.empty(128, 31).bfloat16().cuda())
    with pytest.raises(ValueError):
        gg.backend.gmm(a, b.float(), sizes)
    with pytest.raises(ValueError):
        gg.backend.gmm(a, b, sizes, trans_b=True)
    short = torch.tensor([60, 20])
    with pytest.raises(ValueError):                               # sizes on the host are checked against the operand
        gg.backend.gmm(a, b, short)
    with pytest.raises(ValueError):
        gg.backend.gmm(a, b, torch.tensor([130, -2]))
    with pytest.raises(ValueError):
        gg.backend.gmm(a, a, short, trans_a=True)
    c2 = torch.full((128, 32), 7.0).bfloat16().cuda()             # sizes on the device cannot be: rows past the last
    gg.backend.gmm(a, b, short.cuda(), c=c2)                      # bin are left alone
    assert bool((c2[80:] == 7.0).all()) and rel_err(c2[:80].cpu(), oracle.gmm(a[:80].cpu(), b.cpu(), short)) < TOL


@pytest.mark.parametrize('dtype,k,n', [(torch.bfloat16, 256, 512), (torch.bfloat16, 72, 40), (torch.float32, 64, 64),
                                       (torch.bfloat16, 1 << 16, 64)])
@pytest.mark.parametrize('mode', ['nn', 'nt', 'tn'])
def test_gmm_bins_that_do_not_match_the_operands_stay_in_range(gg, dtype, k, n, mode):
    """Device-side sizes that add up to more rows than the operands have (a stale table), or that are negative:
    the values are then unspecified, but no kernel reads or writes outside the operands -- the rows behind the
    output and a guard region around it keep their canary."""
    if k > 4096 and mode != 'nn':
        pytest.skip('the long-k case exercises the register-staged NN fallback only')
    rows, groups = 700, 4
    a = torch.randn(rows, k, device='cuda').to(dtype)
    if mode == 'tn':
        b = torch.randn(rows, n, device='cuda').to(dtype)
        shape = (groups, k, n)
    else:
        b = torch.randn(groups, n, k, device='cuda').to(dtype) if mode == 'nt' else torch.randn(groups, k, n, device='cuda').to(dtype)
        shape = (rows, n)
    numel = shape[0] * shape[1] * (shape[2] if len(shape) == 3 else 1)
    for sizes in ([300, 300, 300, 300], [900, 0, 0, 0], [200, -50, 400, 5000], [-7, 2000, -2000, 100]):
        guard = 4096
        buf = torch.full((numel + 2 * guard,), 3.0, device='cuda', dtype=dtype)
        c = buf[guard:guard + numel].view(shape)
        gg.backend.gmm(a, b, torch.tensor(sizes, dtype=torch.int32, device='cuda'), trans_a=mode == 'tn', trans_b=mode == 'nt', c=c)
        torch.cuda.synchronize()
        assert bool((buf[:guard] == 3.0).all()) and bool((buf[guard + numel:] == 3.0).all())
    # a table that does match still gives the product
    good = torch.tensor([100, 0, 250, 350], dtype=torch.int32, device='cuda')
    got = gg.backend.gmm(a, b, good, trans_a=mode == 'tn', trans_b=mode == 'nt')
    assert rel_err(got.float(), _ref_gpu(a, b, good.cpu(), mode == 'tn', mode == 'nt')) < TOL


BIG = [  # name, groups, rows, hidden, ffn, skew
    ('gpt2-64e', 64, 16384, 1024, 4096, False),
    ('mixtral', 8, 16384, 4096, 14336, False),
    ('finegrained-zipf', 64, 32768, 2048, 1408, True),
    ('sparse-padded', 16, 12288, 2048, 8192, False),
]


@pytest.mark.parametrize('name,groups,rows,hidden,ffn,skew', BIG)
def test_gmm_benchmark_shapes_vs_fp32(gg, name, groups, rows, hidden, ffn, skew):
    torch.manual_seed(1)
    if skew:
        p = torch.arange(1, groups + 1).float() ** -1.2
        p[-4:] = 0                                               # four experts receive nothing
        sizes = torch.bincount(torch.multinomial(p, rows, replacement=True), minlength=groups)
    else:
        sizes = _sizes(groups, rows, seed=3)
    x = torch.randn(rows, hidden, device='cuda').bfloat16()
    w = (torch.randn(groups, ffn, hidden, device='cuda') * 0.02).bfloat16()
    h = gg.backend.gmm(x, w, sizes, trans_b=True)                               # NT
    ref = _ref_gpu(x, w, sizes, False, True)
    assert rel_err(h, ref) < TOL and max_block_err(h, ref) < 2 * TOL
    y = gg.backend.gmm(h, w, sizes)                                             # NN
    ref = _ref_gpu(h, w, sizes, False, False)
    assert rel_err(y, ref) < TOL and max_block_err(y, ref) < 2 * TOL
    dw = gg.backend.gmm(h, x, sizes, trans_a=True)                              # TN
    ref = _ref_gpu(h, x, sizes, True, False)
    assert rel_err(dw, ref) < TOL and max_block_err(dw, ref) < 2 * TOL
    for e, s in enumerate(sizes.tolist()):
        if s == 0:
            assert torch.count_nonzero(dw[e]) == 0


def test_gmm_autograd(gg):
    sizes = torch.tensor([300, 0, 212])
    a = torch.randn(512, 256, device='cuda').bfloat16().requires_grad_(True)
    b = (torch.randn(3, 128, 256, device='cuda') * 0.1).bfloat16().requires_grad_(True)
    gout = torch.randn(512, 128, device='cuda').bfloat16()
    gg.ops.gmm(a, b, sizes, True).backward(gout)
    af, bf = a.detach().float().requires_grad_(True), b.detach().float().requires_grad_(True)
    outs, start = [], 0
    for e, n in enumerate(sizes.tolist()):
        outs.append(af[start:start + n] @ bf[e].t())
        start += n
    torch.cat(outs).backward(gout.float())
    assert rel_err(a.grad, af.grad) < TOL and rel_err(b.grad, bf.grad) < TOL
    assert torch.count_nonzero(b.grad[1]) == 0


def test_gelu_backward_inplace():
    from megablocks_amd.layers.gelu import gelu_backward_
    for dtype in (torch.bfloat16, torch.float16, torch.float32):
        for shape in ((1000, 257), (1003,), (5,)):            # whole 16-byte vectors; a tail; less than one vector
            x = torch.randn(*shape).to(dtype)
            g = torch.randn(*shape).to(dtype)
            want = oracle.gelu_tanh_backward(g.float(), x.float())
            gd = g.cuda()
            out = gelu_backward_(gd, x.cuda())
            assert out is gd and rel_err(gd.cpu().float(), want) < (1e-5 if dtype == torch.float32 else 1e-2)
        # buffers that are not 16-byte aligned: element by element, same values
        x, g = torch.randn(4100).to(dtype), torch.randn(4100).to(dtype)
        aligned = gelu_backward_(g.cuda()[8:].clone(), x.cuda()[8:].clone())
        base = g.cuda()
        gelu_backward_(base[1:], x.cuda()[1:])
        assert torch.equal(base[8:], aligned) and torch.equal(base[:1].cpu(), g[:1])


DMA_EDGE = [  # groups, rows, k, n: shapes that take the direct-to-LDS kernels, off every tile boundary
    (3, 700, 64, 8), (5, 1030, 128, 264), (2, 255, 192, 1408), (7, 3001, 320, 520), (1, 257, 64, 248),
    (4, 513, 1024, 72), (6, 40, 64, 40),
]


@pytest.mark.parametrize('groups,rows,k,n', DMA_EDGE)
@pytest.mark.parametrize('mode', ['nn', 'nt', 'tn'])
def test_gmm_ragged_shapes_on_the_pipelined_path(gg, groups, rows, k, n, mode):
    sizes = _sizes(groups, rows, seed=rows, empty=(0,) if groups > 2 else ())
    a = torch.randn(rows, k).bfloat16()
    if mode == 'tn':
        b = torch.randn(rows, n).bfloat16()
    elif mode == 'nt':
        b = (torch.randn(groups, n, k) * 0.1).bfloat16()
    else:
        b = (torch.randn(groups, k, n) * 0.1).bfloat16()
    want = oracle.gmm(a, b, sizes, trans_a=mode == 'tn', trans_b=mode == 'nt')
    guard = torch.full((want.numel() + 4096,), 3.0).bfloat16().cuda()       # canary around the output
    c = guard[2048:2048 + want.numel()].view(want.shape)
    got = gg.backend.gmm(a.cuda(), b.cuda(), sizes, trans_a=mode == 'tn', trans_b=mode == 'nt', c=c)
    assert rel_err(got.cpu(), want) < TOL
    assert bool((guard[:2048] == 3.0).all()) and bool((guard[2048 + want.numel():] == 3.0).all())
    if mode == 'tn':
        for e, s in enumerate(sizes.tolist()):
            if s == 0:
                assert torch.count_nonzero(got[e]) == 0


SCHEDULES = [  # name, groups, rows, k, n: one case per branch of the device-side tile schedulers
    ('more than 64 experts, small tile', 80, 24000, 128, 512),
    ('more than 64 experts, big tile', 72, 28800, 128, 768),
    ('fewer tiles than compute units, cut in halves', 2, 1000, 256, 2048),
    ('last round more than half full, not cut', 4, 6400, 128, 2048),
    ('several full rounds and a cut tail', 8, 9000, 64, 2048),
    ('TN with two tiles per workgroup', 4, 3000, 512, 768),
    ('one row per expert', 64, 64, 64, 256),
    ('256 experts: four per lane of the tile table', 256, 40000, 128, 512),
    ('300 experts: five per lane, the last lanes empty', 300, 30000, 64, 264),
    ('65 experts: two per lane', 65, 9000, 192, 512),
]


@pytest.mark.parametrize('name,groups,rows,k,n', SCHEDULES)
def test_gmm_tile_schedules(gg, name, groups, rows, k, n):
    sizes = _sizes(groups, rows, seed=groups + rows, empty=(1,) if groups > 2 else ())
    torch.manual_seed(groups)
    a = torch.randn(rows, k, device='cuda').bfloat16()
    b_nt = (torch.randn(groups, n, k, device='cuda') * 0.1).bfloat16()
    b_nn = (torch.randn(groups, k, n, device='cuda') * 0.1).bfloat16()
    b_tn = torch.randn(rows, n, device='cuda').bfloat16()
    for b, ta, tb in ((b_nt, False, True), (b_nn, False, False), (b_tn, True, False)):
        got = gg.backend.gmm(a, b, sizes, trans_a=ta, trans_b=tb)
        ref = _ref_gpu(a, b, sizes, ta, tb)
        assert rel_err(got, ref) < TOL and max_block_err(got, ref) < 2 * TOL, (name, ta, tb)
        again = gg.backend.gmm(a, b, sizes.cuda().int(), trans_a=ta, trans_b=tb)
        assert torch.equal(again, got)                              # same schedule, same summation order: bit-identical


SPLIT_TAILS = [  # row tiles, column tiles, k (per operand pair): the tail of `row tiles x column tiles` tiles on 256
    # compute units is cut along the reduction into min(256 // tail, 8, K tiles // 8) parts
    (12, 1, 1024),    # 12 tiles, 16 K tiles: two parts
    (12, 1, 4096),    # eight parts
    (68, 16, 1024),   # four full rounds and 64 tiles: four parts (the shape of a Mixtral-sized second product, shorter)
    (85, 1, 768),     # three parts; with two operand pairs the middle one straddles the change of pairs
    (51, 1, 1280),    # five parts
    (36, 1, 1792),    # seven parts
    (3, 43, 640),     # 129 tiles: more than half a round, not cut
    (64, 5, 512),     # a whole round and 64 tiles, reductions too short to cut (8 K tiles): half-height tiles
]


@pytest.mark.parametrize('row_tiles,col_tiles,k', SPLIT_TAILS)
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_gmm_tail_cut_along_the_reduction(gg, row_tiles, col_tiles, k, dtype):
    """NN products whose last round of workgroups is at most half full compute its tiles in parts along K, summed through
    the workspace in a fixed order (mbx_gmm_ws): against fp32, block by block; bit-identical from run to run; the
    workspace's counters are zero again afterwards; without workspace the same values to rounding of the sums' order."""
    from megablocks_amd import _lib
    groups, n = 4, 256 * col_tiles
    per = [256 * (row_tiles // groups)] * groups
    per[0] += 256 * (row_tiles % groups) - 100                       # a ragged last row tile in one expert
    if per[2] >= 256:
        per[2] -= 256
        per[3] += 256
    sizes = torch.tensor(per, dtype=torch.int64)
    rows = int(sizes.sum())
    torch.manual_seed(row_tiles * 100 + col_tiles)
    a = torch.randn(rows, k, device='cuda').to(dtype)
    b = (torch.randn(groups, k, n, device='cuda') * 0.1).to(dtype)
    a2 = torch.randn(rows, k, device='cuda').to(dtype)
    b2 = (torch.randn(groups, k, n, device='cuda') * 0.1).to(dtype)
    ref = _ref_gpu(a, b, sizes, False, False)
    ref2 = ref + _ref_gpu(a2, b2, sizes, False, False)
    guard = torch.full((rows + 64, n), 7.0, device='cuda', dtype=dtype)
    got = gg.backend.gmm(a, b, sizes)
    assert rel_err(got, ref) < TOL and max_block_err(got, ref) < 2 * TOL
    got2 = gg.gmm_dual(a, b, a2, b2, sizes)
    assert rel_err(got2, ref2) < TOL and max_block_err(got2, ref2) < 2 * TOL
    for _ in range(3):
        assert torch.equal(gg.backend.gmm(a, b, sizes), got) and torch.equal(gg.gmm_dual(a, b, a2, b2, sizes), got2)
    ws = gg._workspaces[(torch.cuda.current_device(), _lib.stream().value)]
    assert int(ws[:4096].count_nonzero()) == 0                      # every launch leaves the counters as it found them
    assert bool((guard == 7.0).all())
    # the C ABI without a workspace: one workgroup per tile (or half tile)
    bins = torch.cumsum(sizes, 0).int().cuda()
    plain = torch.empty_like(got)
    _lib.check(_lib.lib.mbx_gmm(_lib.ptr(a), _lib.ptr(b), _lib.ptr(plain), _lib.dtype_of(a), _lib.ptr(bins), groups, rows, k, n,
                                _lib.NN, _lib.stream()))
    assert rel_err(plain, ref) < TOL and rel_err(plain.float(), got.float()) < 2e-3
    # a workspace too small for two parts per tail tile, or misaligned: ignored
    small = torch.zeros(4096 + 100, dtype=torch.uint8, device='cuda')
    out = torch.empty_like(got)
    _lib.check(_lib.lib.mbx_gmm_ws(_lib.ptr(a), _lib.ptr(b), None, None, _lib.ptr(out), _lib.dtype_of(a), _lib.ptr(bins), groups,
                                   rows, k, n, _lib.NN, _lib.ptr(small), small.numel(), _lib.stream()))
    assert torch.equal(out, plain)
    assert _lib.lib.mbx_gmm_ws(_lib.ptr(a), _lib.ptr(b), _lib.ptr(a2), None, _lib.ptr(out), _lib.dtype_of(a), _lib.ptr(bins), groups,
                               rows, k, n, _lib.NN, None, 0, _lib.stream()) == _lib.EINVAL


@pytest.mark.parametrize('column_tiles,k_tiles,cut', [(20, 79, False), (20, 80, True), (24, 159, False), (24, 160, True)])   # tails of 64 and 128 tiles: four parts, two
def test_gmm_tail_behind_full_rounds_is_cut_along_long_reductions_only(gg, monkeypatch, column_tiles, k_tiles, cut):
    """Sixteen row tiles: a full round and a tail.  Not cut, the launch computes what it does without a workspace, to the bit; cut, another order of the sums."""
    sizes, k, n = torch.tensor([1024] * 4), 64 * k_tiles, 256 * column_tiles
    torch.manual_seed(k_tiles)
    a = torch.randn(4096, k, device='cuda').bfloat16()
    b = torch.empty(4, k, n, device='cuda', dtype=torch.bfloat16).normal_(0, k ** -0.5)
    got = gg.gmm(a, b, sizes)
    ref = _ref_gpu(a, b, sizes, False, False)
    assert rel_err(got, ref) < TOL and max_block_err(got, ref) < 2 * TOL
    monkeypatch.setattr(gg, 'GMM_WORKSPACE', False)
    assert torch.equal(gg.gmm(a, b, sizes), got) != (cut and _units() == 256)


MIXED_ROWS = [  # per-expert row counts around the boundaries between full (256-row) and half-height (128-row) tiles
    [256, 257, 300, 384, 385, 129, 128, 1, 0, 512, 640, 127],
    [300] * 48,                       # full and half-height tiles alternate along the tile list, several rounds
    [260, 250] * 40,                  # more than 64 experts
    [130] * 64,                       # on average below the full tile: half-height tiles only
    [2048 + 37 * (i % 5) for i in range(8)] + [100, 2100, 0, 385],     # many full tiles, a few short last ones
    [(300, 0, 700, 256, 40)[i % 5] for i in range(150)],             # short last tiles with several experts per lane
]


@pytest.mark.parametrize('rows_per_expert', MIXED_ROWS, ids=lambda r: f'{len(r)}experts')
@pytest.mark.parametrize('k,n', [(256, 1024), (512, 264)])
def test_gmm_full_and_half_height_row_tiles(gg, rows_per_expert, k, n):
    sizes = torch.tensor(rows_per_expert, dtype=torch.int64)
    groups, rows = len(rows_per_expert), int(sizes.sum())
    torch.manual_seed(rows)
    a = torch.randn(rows, k, device='cuda').bfloat16()
    b_nt = (torch.randn(groups, n, k, device='cuda') * 0.1).bfloat16()
    b_nn = (torch.randn(groups, k, n, device='cuda') * 0.1).bfloat16()
    for b, tb in ((b_nt, True), (b_nn, False)):
        got = gg.backend.gmm(a, b, sizes, trans_b=tb)
        ref = _ref_gpu(a, b, sizes, False, tb)
        assert rel_err(got, ref) < TOL and max_block_err(got, ref) < 2 * TOL, tb
    a2 = torch.randn(rows, k, device='cuda').bfloat16()
    b2 = (torch.randn(groups, k, n, device='cuda') * 0.1).bfloat16()
    got = gg.gmm_dual(a, b_nn, a2, b2, sizes)
    ref = _ref_gpu(a, b_nn, sizes, False, False).float() + _ref_gpu(a2, b2, sizes, False, False).float()
    assert rel_err(got.float(), ref) < TOL


@pytest.mark.parametrize('k', [264, 384, 392, 648, 1408])      # k mod 256 = 8, 128, 136, 136, 128: the last row of tiles
@pytest.mark.parametrize('n', [256, 520])                      # is half-height up to 128 rows, full above
def test_gmm_tn_last_row_of_tiles(gg, k, n):
    sizes = torch.tensor([700, 0, 64, 3000, 1, 331])
    rows = int(sizes.sum())
    torch.manual_seed(k + n)
    a = torch.randn(rows, k, device='cuda').bfloat16()
    b = torch.randn(rows, n, device='cuda').bfloat16()
    ref = _ref_gpu(a, b, sizes, True, False)
    guard = torch.full((ref.numel() + 4096,), 3.0, device='cuda').bfloat16()
    c = guard[2048:2048 + ref.numel()].view(ref.shape)
    got = gg.backend.gmm(a, b, sizes, trans_a=True, c=c)
    assert rel_err(got, ref) < TOL and max_block_err(got, ref) < 2 * TOL
    assert torch.count_nonzero(got[1]) == 0
    assert bool((guard[:2048] == 3.0).all()) and bool((guard[2048 + ref.numel():] == 3.0).all())


# Short reductions whose experts load the XCDs alike are dealt to XCDs as whole experts (the kernel decides from the
# row counts): equal experts, equal experts next to empty ones, a count that is no multiple of eight (never balanced:
# an eighth of every expert per XCD, as for long reductions), nearly equal ones, and one XCD's worth of experts.
WHOLE_EXPERTS = [[200] * 16, [256, 0] * 8, [320] * 12, [250 + (7 * i) % 13 for i in range(64)], [192] * 8, [64] * 40 + [0] * 24]


@pytest.mark.parametrize('rows_per_expert', WHOLE_EXPERTS, ids=lambda r: f'{len(r)}x{r[0]}')
@pytest.mark.parametrize('k,n', [(1024, 512), (264, 1032), (128, 256)])
def test_gmm_tn_short_reductions_dealt_by_expert(gg, rows_per_expert, k, n):
    sizes = torch.tensor(rows_per_expert)
    rows = int(sizes.sum())
    torch.manual_seed(rows + k)
    a = torch.randn(rows, k, device='cuda').bfloat16()
    b = torch.randn(rows, n, device='cuda').bfloat16()
    ref = _ref_gpu(a, b, sizes, True, False)
    guard = torch.full((ref.numel() + 4096,), 3.0, device='cuda').bfloat16()
    c = guard[2048:2048 + ref.numel()].view(ref.shape)
    got = gg.backend.gmm(a, b, sizes.cuda(), trans_a=True, c=c)
    assert rel_err(got, ref) < TOL and max_block_err(got, ref) < 2 * TOL
    for e, r in enumerate(rows_per_expert):
        if r == 0:
            assert torch.count_nonzero(got[e]) == 0
    assert bool((guard[:2048] == 3.0).all()) and bool((guard[2048 + ref.numel():] == 3.0).all())


def _random_shapes(count, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda lo, hi: int(torch.randint(lo, hi + 1, (1,), generator=g))
    shapes = []
    for i in range(count):
        groups, rows = r(1, 70), r(1, 5000)
        if i % 3 == 0:      # the pipelined kernels: k a multiple of 64
            k, n = 64 * r(1, 17), 8 * r(1, 140)
        elif i % 3 == 1:    # the register-staged kernels: multiples of 8
            k, n = 8 * r(1, 140), 8 * r(1, 140)
        else:               # anything
            k, n = r(1, 600), r(1, 600)
        shapes.append((groups, rows, k, n))
    return shapes


@pytest.mark.parametrize('groups,rows,k,n', _random_shapes(36, seed=7))
def test_gmm_random_shapes_with_canaries(gg, groups, rows, k, n):
    sizes = _sizes(groups, rows, seed=groups * 7 + rows, empty=(0,) if groups > 3 else ())
    torch.manual_seed(rows)
    a = torch.randn(rows, k, device='cuda').bfloat16()
    for mode in ('nn', 'nt', 'tn'):
        if mode == 'tn':
            b = torch.randn(rows, n, device='cuda').bfloat16()
        else:
            b = (torch.randn((groups, n, k) if mode == 'nt' else (groups, k, n), device='cuda') * 0.1).bfloat16()
        ref = _ref_gpu(a, b, sizes, mode == 'tn', mode == 'nt')
        guard = torch.full((ref.numel() + 4096,), 3.0, device='cuda').bfloat16()       # canary around the output
        c = guard[2048:2048 + ref.numel()].view(ref.shape)
        got = gg.backend.gmm(a, b, sizes, trans_a=mode == 'tn', trans_b=mode == 'nt', c=c)
        assert rel_err(got, ref) < TOL and max_block_err(got, ref) < 2 * TOL, mode
        assert bool((guard[:2048] == 3.0).all()) and bool((guard[2048 + ref.numel():] == 3.0).all()), mode


DUAL = [  # groups, rows, k, n, single launch expected
    (8, 4000, 512, 1024, True), (3, 700, 256, 264, True), (64, 16384, 1408, 2048, True), (70, 21000, 256, 512, True),
    (4, 1000, 192, 256, False), (2, 300, 100, 36, False), (1, 64, 256, 8, True),
]


@pytest.mark.parametrize('groups,rows,k,n,single', DUAL)
@pytest.mark.parametrize('trans_b', [False, True])
def test_gmm_dual_is_the_sum_of_two_products(gg, groups, rows, k, n, single, trans_b):
    from megablocks_amd import _lib
    sizes = _sizes(groups, rows, seed=rows + k, empty=(1,) if groups > 2 else ())
    torch.manual_seed(k)
    a, a2 = (torch.randn(rows, k, device='cuda').bfloat16() for _ in range(2))
    shape = (groups, n, k) if trans_b else (groups, k, n)
    b, b2 = ((torch.randn(shape, device='cuda') * 0.1).bfloat16() for _ in range(2))
    ref = _ref_gpu(a, b, sizes, False, trans_b) + _ref_gpu(a2, b2, sizes, False, trans_b)
    _lib.profile_hook = []
    try:
        got = gg.gmm_dual(a, b, a2, b2, sizes, trans_b=trans_b)
        names = [r[0] for r in _lib.profile_hook]
    finally:
        _lib.profile_hook = None
    assert (names == ['gmm_nt_dual' if trans_b else 'gmm_nn_dual']) == single   # else: two products and a sum
    assert got.dtype == torch.bfloat16 and rel_err(got, ref) < TOL and max_block_err(got, ref) < 2 * TOL
    c = torch.full((rows, n), 5.0, device='cuda').bfloat16()
    assert gg.gmm_dual(a, b, a2, b2, sizes.cuda().int(), trans_b=trans_b, c=c) is c and torch.equal(c, got)
    with pytest.raises(ValueError):
        gg.gmm_dual(a, b, a2[:, :-8], b2, sizes, trans_b=trans_b)


def _ref_in_pieces(check, a, b, sizes, trans_a, trans_b, got):
    """Compare `got` with the fp32 product expert by expert (an fp32 copy of a whole operand of several GiB
    at once is not needed then); `check(piece_of_got, reference_piece)`."""
    start = 0
    for e, n in enumerate(sizes.tolist()):
        ae = a[start:start + n].float()
        if trans_a and n:
            check(got[e], ae.t() @ b[start:start + n].float())
        elif n:
            check(got[start:start + n], ae @ (b[e].float().t() if trans_b else b[e].float()))
        start += n


LARGE = [  # name, rows per expert, k, n: the [rows, k] or the [rows, n] matrix (or one expert's share of it) of 2 .. 5 GiB
    ('rows-by-k-2.3GiB', [150000, 0, 100000, 50000], 4096, 256),
    ('rows-by-n-2.3GiB', [150000, 0, 100000, 50000], 256, 4096),
    ('one-expert-4.3GiB-of-4.6GiB', [20000, 560000, 20], 4096, 128),
]


@pytest.mark.parametrize('name,rows_per_expert,k,n', LARGE, ids=[c[0] for c in LARGE])
def test_gmm_operands_beyond_2GiB(gg, name, rows_per_expert, k, n):
    """Byte offsets inside the big matrices pass 2^31 and 2^32: same kernels, same tolerance."""
    from megablocks_amd import _lib
    sizes = torch.tensor(rows_per_expert)
    rows, groups = int(sizes.sum()), len(rows_per_expert)
    torch.manual_seed(rows % 1000)
    a = torch.empty(rows, k, device='cuda', dtype=torch.bfloat16).normal_()
    a2 = a.flip(0)
    w_nn = torch.empty(groups, k, n, device='cuda', dtype=torch.bfloat16).normal_(std=0.1)
    w_nt = torch.empty(groups, n, k, device='cuda', dtype=torch.bfloat16).normal_(std=0.1)
    b_tn = torch.empty(rows, n, device='cuda', dtype=torch.bfloat16).normal_()
    assert max(a.numel(), b_tn.numel()) * 2 >= 2 ** 31

    def check(got, ref):
        assert rel_err(got, ref) < TOL and max_block_err(got, ref, bm=256, bn=256) < 2 * TOL

    _lib.profile_hook = []
    try:
        nn = gg.backend.gmm(a, w_nn, sizes)
        nt = gg.backend.gmm(a, w_nt, sizes, trans_b=True)
        tn = gg.backend.gmm(a, b_tn, sizes, trans_a=True)
        dual = gg.gmm_dual(a, w_nn, a2, w_nn, sizes) if k >= 256 else None
        names = [r[0] for r in _lib.profile_hook]
    finally:
        _lib.profile_hook = None
    _ref_in_pieces(check, a, w_nn, sizes, False, False, nn)
    _ref_in_pieces(check, a, w_nt, sizes, False, True, nt)
    _ref_in_pieces(check, a, b_tn, sizes, True, False, tn)
    assert torch.count_nonzero(tn[[i for i, s in enumerate(rows_per_expert) if s == 0]]) == 0
    if dual is not None:
        assert names[-1] == 'gmm_nn_dual'            # one launch, not two products and a sum
        second = gg.backend.gmm(a2, w_nn, sizes)
        _ref_in_pieces(check, a2, w_nn, sizes, False, False, second)
        assert rel_err(dual, nn.float() + second.float()) < TOL


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize('act_name', ['silu', 'gelu_tanh'])
def test_fused_gated_activation_matches_the_two_step_formulation(dtype, act_name):
    import torch.nn.functional as F
    from megablocks_amd.layers.arguments import DEFAULT_ACTIVATION_FN
    from megablocks_amd.layers.glu import gated_activation
    fn = F.silu if act_name == 'silu' else DEFAULT_ACTIVATION_FN
    a = (torch.randn(777, 1408) * 2).to(dtype).cuda().requires_grad_(True)
    b = torch.randn(777, 1408).to(dtype).cuda().requires_grad_(True)
    g = torch.randn(777, 1408).to(dtype).cuda()
    out = gated_activation(fn, a, b)
    out.backward(g)
    a2, b2 = a.detach().clone().requires_grad_(True), b.detach().clone().requires_grad_(True)
    want = fn(a2) * b2                                   # the reference's two element-wise ops (glu.py:89)
    want.backward(g)
    tol = 1e-6 if dtype == torch.float32 else 1e-2
    assert rel_err(out, want) < tol and rel_err(a.grad, a2.grad) < tol and rel_err(b.grad, b2.grad) < tol
    if dtype != torch.float32:                           # forward: same roundings -> almost always the same bits
        assert float((out != want).float().mean()) < 1e-3
    wantf = fn(a.detach().float().cpu()) * b.detach().float().cpu()      # CPU fp32 check of the math itself
    assert rel_err(out.cpu(), wantf) < (1e-5 if dtype == torch.float32 else 1e-2)
    odd = torch.randn(5, 3).to(dtype).cuda()             # not a multiple of 16 bytes: plain torch ops
    assert torch.equal(gated_activation(fn, odd, odd), fn(odd) * odd)


EPILOGUE = [  # groups, rows, k, n -- full and half-height tiles, partial last column tile, shapes off the fused path
    (8, 4096, 1024, 4096), (64, 16384, 1024, 1024), (5, 1500, 320, 264), (3, 700, 128, 1408), (1, 37, 64, 8),
    (4, 1000, 72, 256), (16, 6000, 2048, 520), (72, 5000, 128, 264),
]


@pytest.mark.parametrize('groups,rows,k,n', EPILOGUE)
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16, torch.float32])
def test_gmm_with_activation_epilogues(gg, groups, rows, k, n, dtype):
    """gmm_act: (x @ w1^T, gelu_tanh of it) in one launch; gmm_dact: round(dy @ w2^T) * gelu_tanh'(pre).  Against the
    two-step formulation of mlp.py:521-522 and mlp.py:478-483 / gelu.py:9-13 in fp32 with the reference's roundings."""
    torch.manual_seed(groups * 7 + n)
    sizes = _sizes(groups, rows, seed=rows + k, empty=(1,) if groups > 2 else ())
    a = torch.randn(rows, k, device='cuda').to(dtype)
    b = (torch.randn(groups, n, k, device='cuda') * (1.5 / k ** 0.5)).to(dtype)      # pre-activations of order one
    ref = _ref_gpu(a, b, sizes, False, True)
    want_pre = ref.to(dtype)
    want_act = torch.nn.functional.gelu(want_pre.float(), approximate='tanh')
    guard = torch.full((rows + 64, n), 5.0, device='cuda', dtype=dtype)
    pre, act = gg.gmm_act(a, b, sizes, fuse=True)
    assert pre.shape == (rows, n) and act.shape == (rows, n) and pre.dtype == dtype and act.dtype == dtype
    tol = 1e-4 if dtype == torch.float32 else TOL
    assert rel_err(pre.float(), ref) < tol
    assert torch.equal(pre, gg.backend.gmm(a, b, sizes, trans_b=True))         # the product itself is the same kernel's
    # the activation is taken of the stored product: one rounding step of the output type away from the fp32 formula
    assert rel_err(act.float(), torch.nn.functional.gelu(pre.float(), approximate='tanh')) < (1e-6 if dtype == torch.float32 else 3e-3)
    assert rel_err(act.float(), want_act) < tol

    dy = torch.randn(rows, k, device='cuda').to(dtype)
    x_pre = (torch.randn(rows, n, device='cuda') * 1.5).to(dtype)
    prod = _ref_gpu(dy, b, sizes, False, True).to(dtype).float()
    want = prod * oracle.gelu_tanh_backward(torch.ones_like(prod).cpu(), x_pre.float().cpu()).cuda()
    got = gg.gmm_dact(dy, b, x_pre, sizes, fuse=True)
    assert got.shape == (rows, n) and got.dtype == dtype and rel_err(got.float(), want) < tol
    out = guard[:rows]
    assert gg.gmm_dact(dy, b, x_pre, sizes, c=out, fuse=True) is out and torch.equal(out, got)
    two_step = gg.gmm_dact(dy, b, x_pre, sizes, fuse=False)            # product, then gelu_backward_ in place
    assert rel_err(two_step.float(), want) < tol and rel_err(got.float(), two_step.float()) < (1e-6 if dtype == torch.float32 else 4e-3)
    pre2, act2 = gg.gmm_act(a, b, sizes, fuse=False)
    assert torch.equal(pre2, pre) and rel_err(act.float(), act2.float()) < (1e-6 if dtype == torch.float32 else 4e-3)
    assert bool((guard[rows:] == 5.0).all())
    with pytest.raises(ValueError):
        gg.gmm_dact(dy, b, x_pre, sizes, c=x_pre)                              # the epilogue reads pre while it writes c
    with pytest.raises(ValueError):
        gg.gmm_act(a, b[:, :, :k - 8].contiguous(), sizes)


@pytest.mark.parametrize('k', [64, 72])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_gelu_epilogues_on_every_16_bit_value(gg, dtype, k):
    """gelu_tanh and its derivative in the epilogues at every finite 16-bit value of the pre-activation (the product itself is
    exactly 1, or the value): finite wherever the separate pass is, within a rounding step of the function in fp64, and
    no more of them off the nearest 16-bit value than the separate pass has."""
    x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype).cuda()
    x = torch.where(torch.isfinite(x), x, torch.zeros_like(x)).view(256, 256)
    x64 = x.double()
    u = math.sqrt(2 / math.pi) * (x64 + 0.044715 * x64 ** 3)
    q = 2 * math.sqrt(2 / math.pi) * (1 + 3 * 0.044715 * x64 ** 2)
    tail = x64.abs() > 40     # there the derivative is 0 or 1 in any type
    want_grad = torch.where(tail, (x64 > 0).double(), torch.sigmoid(2 * u) * (1 + x64 * torch.sigmoid(-2 * u) * q))
    ones, rows = torch.zeros(256, k, device='cuda', dtype=dtype), torch.tensor([256], device='cuda')
    ones[:, 0] = 1
    values = torch.zeros(256, 256, k, device='cuda', dtype=dtype)
    values[:, :, 0] = x
    # a sigmoid below the normal fp32 range (2^-126) counts as zero; the derivative's other factor is below 2^8 there
    step, least = torch.finfo(dtype).eps, max(torch.finfo(dtype).tiny * torch.finfo(dtype).eps, 2.0 ** -118)

    def check(got, separate, want):
        there = torch.isfinite(separate) & torch.isfinite(want.to(dtype))
        assert bool(torch.isfinite(got[there]).all())
        d = (got[there].double() - want[there]).abs()
        # one step of the result; of 1 where the derivative crosses zero (its two terms are rounded in fp32: 2^-22 each)
        assert bool((d <= step * want[there].abs() + torch.clamp(2.0 ** -21 * (x64[there].abs() < 2), min=least)).all())
        assert int((got[there] != want[there].to(dtype)).sum()) <= int((separate[there] != want[there].to(dtype)).sum())
    dact = [gg.gmm_dact(ones, ones[None], x, rows, fuse=fuse) for fuse in (True, False)]
    check(*dact, want_grad)
    one = torch.ones_like(x)
    dglu = [gg.gmm_dglu(ones, ones[None], x, one, rows, 1, fuse=fuse) for fuse in (True, False)]
    check(dglu[0][0], dglu[1][0], want_grad)
    each = torch.ones(256, dtype=torch.int64, device='cuda')
    check(gg.gmm_act(ones, values, each, fuse=True)[1], gg.gmm_act(ones, values, each, fuse=False)[1], x64 * torch.sigmoid(2 * u))


@pytest.mark.parametrize('groups,rows,k,n', EPILOGUE)
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize('act', [0, 1], ids=['silu', 'gelu_tanh'])
def test_gmm_with_gated_activation_backward_epilogue(gg, groups, rows, k, n, dtype, act):
    """gmm_dglu: with g = round(dy @ w2^T), (round(g x2) act'(x1), g round(act(x1))) in one launch, against autograd's
    gradient of act(x1) * x2 in fp32 (glu.py:120-124,135-153) and against the product followed by the element-wise
    kernel, which it must equal to a rounding step of the output type."""
    from megablocks_amd.layers.glu import _glu_backward
    torch.manual_seed(groups * 11 + n + act)
    sizes = _sizes(groups, rows, seed=rows + k + 1, empty=(1,) if groups > 2 else ())
    dy = torch.randn(rows, k, device='cuda').to(dtype)
    b = (torch.randn(groups, n, k, device='cuda') * (1.0 / k ** 0.5)).to(dtype)
    x1 = (torch.randn(rows, n, device='cuda') * 1.5).to(dtype)
    x2 = torch.randn(rows, n, device='cuda').to(dtype)
    g = _ref_gpu(dy, b, sizes, False, True).to(dtype).float()
    fn = torch.nn.functional.silu if act == 0 else (lambda t: torch.nn.functional.gelu(t, approximate='tanh'))
    a_, b_ = x1.float().requires_grad_(True), x2.float().requires_grad_(True)
    (fn(a_) * b_).backward(g)
    d1, d2 = gg.gmm_dglu(dy, b, x1, x2, sizes, act, fuse=True)
    tol = 1e-4 if dtype == torch.float32 else TOL
    assert d1.shape == (rows, n) and d2.shape == (rows, n) and d1.dtype == dtype and d2.dtype == dtype
    assert rel_err(d1.float(), a_.grad) < tol and rel_err(d2.float(), b_.grad) < tol
    t1, t2 = _glu_backward(gg.backend.gmm(dy, b, sizes, trans_b=True), x1, x2, act)
    step = 1e-6 if dtype == torch.float32 else 4e-3
    assert rel_err(d1.float(), t1.float()) < step and rel_err(d2.float(), t2.float()) < step
    u1, u2 = gg.gmm_dglu(dy, b, x1, x2, sizes.cuda(), act, fuse=False)
    assert torch.equal(u1, t1) and torch.equal(u2, t2)
    with pytest.raises(ValueError):
        gg.gmm_dglu(dy, b, x1[:, :n - 8].contiguous(), x2, sizes, act)


@pytest.mark.parametrize('groups,rows,k,n', EPILOGUE + [(6, 2500, 256, 1416), (2, 300, 64, 136)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize('act', [0, 1], ids=['silu', 'gelu_tanh'])
def test_gmm_with_gated_activation_epilogue(gg, groups, rows, k, n, dtype, act):
    """gmm_glu: (x @ w1^T, x @ v1^T, round(round(act(x1)) x2)) in one launch (glu.py:201-204): both products must be
    the plain kernel's bit for bit, the gated activation within a rounding step of the element-wise kernel's and of the
    fp32 formula on the stored products."""
    from megablocks_amd.layers.glu import _glu_forward
    torch.manual_seed(groups * 13 + n + act)
    sizes = _sizes(groups, rows, seed=rows + k + 2, empty=(1,) if groups > 2 else ())
    a = torch.randn(rows, k, device='cuda').to(dtype)
    w1 = (torch.randn(groups, n, k, device='cuda') * (1.5 / k ** 0.5)).to(dtype)
    v1 = (torch.randn(groups, n, k, device='cuda') * (1.0 / k ** 0.5)).to(dtype)
    guard = torch.full((3, rows + 16, n), 7.0, device='cuda', dtype=dtype)
    x1, x2, h = gg.gmm_glu(a, w1, v1, sizes, act, fuse=True)
    p1, p2 = gg.backend.gmm(a, w1, sizes, trans_b=True), gg.backend.gmm(a, v1, sizes.cuda(), trans_b=True)
    assert x1.shape == (rows, n) and h.shape == (rows, n) and h.dtype == dtype
    assert torch.equal(x1, p1) and torch.equal(x2, p2)
    fn = torch.nn.functional.silu if act == 0 else (lambda t: torch.nn.functional.gelu(t, approximate='tanh'))
    want = fn(p1.float()).to(dtype).float() * p2.float()
    step = 1e-6 if dtype == torch.float32 else 4e-3
    assert rel_err(h.float(), want) < step
    assert rel_err(h.float(), _glu_forward(p1, p2, act).float()) < step
    y1, y2, g = gg.gmm_glu(a, w1, v1, sizes, act, fuse=False)
    assert torch.equal(y1, p1) and torch.equal(y2, p2) and torch.equal(g, _glu_forward(p1, p2, act))
    assert bool((guard == 7.0).all())
    with pytest.raises(ValueError):
        gg.gmm_glu(a, w1, v1[:, :n - 8].contiguous(), sizes, act)


def _routing(tokens, experts, top_k, seed, blocking=0):
    """(indices, bin_ids, bins, padded_bins or None, tokens_per_expert) of a random assignment, from the library's ops."""
    from megablocks_amd import ops
    g = torch.Generator().manual_seed(seed)
    top = torch.randint(0, experts, (tokens * top_k,), generator=g, dtype=torch.int32)
    if experts > 2:
        top[top == 1] = 0                                   # an expert without tokens
    top = top.cuda()
    end_bit = max(int(math.ceil(math.log2(experts))), 1)
    bin_ids, indices = ops.sort(top, end_bit)
    tpe = ops.histogram(top, experts)
    bins = ops.inclusive_cumsum(tpe, 0).view(-1)
    padded_bins = None
    if blocking:
        padded_bins = ops.inclusive_cumsum(ops.round_up(tpe, blocking), 0).view(-1)
    return indices, bin_ids, bins, padded_bins, tpe


GATHERED = [  # tokens, experts, top_k, k, n, blocking
    (4096, 8, 2, 1024, 512, 0), (3000, 5, 1, 320, 264, 0), (700, 3, 4, 128, 1408, 0), (37, 1, 1, 64, 8, 0),
    (2048, 16, 4, 256, 384, 128), (1000, 72, 2, 128, 264, 128), (5000, 64, 1, 1024, 1024, 0), (9, 4, 2, 64, 136, 128),
    (3000, 12, 3, 128, 256, 0), (4000, 64, 6, 192, 1408, 0), (1111, 9, 7, 64, 128, 128), (500, 40, 33, 64, 64, 0),
]


@pytest.mark.parametrize('tokens,experts,top_k,k,n,blocking', GATHERED)
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_gmm_on_rows_gathered_on_the_fly(gg, tokens, experts, top_k, k, n, blocking, dtype):
    """gmm_gather: the first product(s) of the experts reading their rows from the ungathered tokens must equal, bit
    for bit, ops.gather / ops.padded_gather (dmoe.py:219 / :273) followed by gmm, gmm_act and gmm_glu: the same
    products over the same operand values in the same order, only fetched from other addresses."""
    torch.manual_seed(tokens + n)
    indices, bin_ids, bins, padded_bins, tpe = _routing(tokens, experts, top_k, seed=tokens + k, blocking=blocking)
    x = torch.randn(tokens, k, device='cuda').to(dtype)
    w1 = (torch.randn(experts, n, k, device='cuda') * (1.5 / k ** 0.5)).to(dtype)
    v1 = (torch.randn(experts, n, k, device='cuda') * (1.0 / k ** 0.5)).to(dtype)
    rows = tokens * top_k if padded_bins is None else int(padded_bins[-1])
    sizes = tpe if padded_bins is None else torch.diff(padded_bins, prepend=padded_bins.new_zeros(1))
    src = gg.GatheredRows(x, indices, bin_ids, bins, padded_bins, top_k, rows)
    a = src.materialize()
    assert a.shape == (rows, k)
    guard = torch.full((3, rows + 16, n), 7.0, device='cuda', dtype=dtype)
    (c,) = gg.gmm_gather(src, w1, sizes)
    assert torch.equal(c, gg.backend.gmm(a, w1, sizes, trans_b=True))
    c, h = gg.gmm_gather(src, w1, sizes, act=gg.ACT_GELU_TANH)
    want_c, want_h = gg.gmm_act(a, w1, sizes, fuse=True)
    assert torch.equal(c, want_c) and torch.equal(h, want_h)
    # ... and, directly, the CPU oracle's gather (kernels.py:107-170) and grouped product on the same inputs, with the
    # activations of mlp.py:521-522 / glu.py:201-204 applied to the product as stored
    cpu = lambda t: None if t is None else t.cpu()
    if padded_bins is None:
        o_a = oracle.gather(cpu(x), cpu(indices), cpu(bin_ids), None, cpu(bins), top_k)
    else:
        o_a = oracle.padded_gather(cpu(x), cpu(indices), cpu(bin_ids), None, cpu(bins), cpu(padded_bins), top_k)
    assert torch.equal(a.cpu(), o_a)
    o_x1 = oracle.gmm(o_a, cpu(w1), cpu(sizes), trans_b=True)
    o_x2 = oracle.gmm(o_a, cpu(v1), cpu(sizes), trans_b=True)
    gelu = lambda t: torch.nn.functional.gelu(t.float(), approximate='tanh').to(dtype)
    silu = lambda t: torch.nn.functional.silu(t.float()).to(dtype)
    if rows:
        assert rel_err(c.cpu(), o_x1) < TOL and rel_err(h.cpu(), gelu(o_x1)) < TOL
    for act in (0, 1):
        x1, x2, h = gg.gmm_gather(src, w1, sizes, b2=v1, act=act)
        w_x1, w_x2, w_h = gg.gmm_glu(a, w1, v1, sizes, act, fuse=True)
        assert torch.equal(x1, w_x1) and torch.equal(x2, w_x2) and torch.equal(h, w_h)
        if rows:
            o_h = ((silu, gelu)[act](o_x1).float() * o_x2.float()).to(dtype)
            assert rel_err(x1.cpu(), o_x1) < TOL and rel_err(x2.cpu(), o_x2) < TOL and rel_err(h.cpu(), o_h) < TOL
    assert bool((guard == 7.0).all())


COMBINED = [  # tokens (= rows: one expert per token), experts, k, n
    (4096, 8, 1024, 512), (3000, 5, 320, 264), (37, 1, 64, 8), (5000, 64, 1024, 1024), (16384, 64, 512, 1024),
    (700, 3, 128, 1408), (2600, 4, 2048, 256), (300, 40, 64, 136), (511, 2, 1024, 64), (65, 1, 1024, 512), (8192, 100, 1024, 256),
]


@pytest.mark.parametrize('tokens,experts,k,n', COMBINED)
@pytest.mark.parametrize('dtype,w_dtype', [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                           (torch.bfloat16, torch.float32), (torch.float16, torch.float32),
                                           (torch.bfloat16, None)])
def test_gmm_with_the_combine_in_the_epilogue(gg, monkeypatch, tokens, experts, k, n, dtype, w_dtype):
    """gmm_scatter: with one expert per token the experts' second product (mlp.py:523, glu.py:205) writes the layer's
    weighted combine (dmoe.py:280, kernels.py:173-207) from its store phase.  Product and combined output must equal,
    bit for bit, gmm followed by the scatter kernel (the same roundings in the same places), and meet the CPU oracle's
    product and scatter directly; rows of the output that no assignment names are left alone."""
    from megablocks_amd.backend import kernels
    torch.manual_seed(tokens + n)
    indices, bin_ids, bins, _, tpe = _routing(tokens, experts, 1, seed=tokens + k)
    h = torch.randn(tokens, k, device='cuda').to(dtype)
    w2 = (torch.randn(experts, k, n, device='cuda') * (1.5 / k ** 0.5)).to(dtype)
    weights = None if w_dtype is None else (torch.rand(tokens, device='cuda') + 0.25).to(w_dtype)
    combine = gg.CombinedRows(indices, bin_ids, bins, weights)
    monkeypatch.setattr(gg, 'GMM_WORKSPACE', False)   # the plain product without a tail cut along K, as the combined launch computes it
    want_y = gg.backend.gmm(h, w2, tpe)
    want_out = kernels.scatter(want_y, indices, bin_ids, weights, bins, 1)
    y, out = gg.gmm_scatter(h, w2, tpe, combine)
    assert torch.equal(y, want_y) and torch.equal(out, want_out)
    y2, out2 = gg.gmm_scatter(h, w2, tpe, combine, keep_product=False)
    assert torch.equal(out2, want_out) and (y2 is None or torch.equal(y2, want_y))
    cpu = lambda t: None if t is None else t.cpu()
    o_y = oracle.gmm(cpu(h), cpu(w2), cpu(tpe))
    o_out = oracle.scatter(o_y, cpu(indices), cpu(bin_ids), cpu(weights), cpu(bins), 1)
    assert rel_err(y.cpu(), o_y) < TOL and rel_err(out.cpu(), o_out) < TOL
    # assignments outside the tokens, and a token nobody names: those rows are not combined, that row is not written
    bad = indices.clone()
    bad[::5] = -3
    bad[2::7] = tokens + 11
    lib, _lib = gg.lib, gg._lib
    canvas = torch.full((tokens, n), 3.0, device='cuda', dtype=dtype)
    dbins = tpe.cumsum(0).int()
    rc = lib.mbx_gmm_scatter(_lib.ptr(h), _lib.ptr(w2), None, _lib.ptr(canvas), _lib.dtype_of(h), _lib.ptr(dbins), experts,
                             tokens, k, n, _lib.ptr(bad), _lib.ptr(weights), 0 if weights is None else _lib.dtype_of(weights),
                             tokens, _lib.stream())
    if k % 64 == 0 and n % 8 == 0:
        assert rc == 0
        keep = (bad >= 0) & (bad < tokens)
        want = torch.full_like(canvas, 3.0)
        want[bad[keep].long()] = want_out[indices[keep].long()]    # the rows that kept their assignment
        assert torch.equal(canvas, want)
    else:
        assert rc == _lib.EUNSUPPORTED


GATHERED_TN = [  # tokens, experts, top_k, hidden of the tokens (n), columns of the other operand (k), blocking
    (4096, 8, 2, 1024, 512, 0), (3000, 5, 1, 320, 264, 0), (700, 3, 4, 128, 1408, 0), (2048, 16, 4, 256, 384, 128),
    (1000, 72, 2, 128, 264, 128), (5000, 64, 1, 1024, 1024, 0), (9, 4, 2, 64, 136, 128), (4000, 64, 6, 192, 1408, 0),
    (1111, 9, 7, 64, 256, 128), (500, 40, 33, 64, 192, 0), (2500, 4, 2, 2048, 320, 0),
]


@pytest.mark.parametrize('tokens,experts,top_k,n,k,blocking', GATHERED_TN)
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_gmm_weight_gradient_on_rows_gathered_on_the_fly(gg, tokens, experts, top_k, n, k, blocking, dtype):
    """gmm_tn_gather: the weight gradient d^T @ x_gathered of the experts' first product (mlp.py:485-491, glu.py:154-159)
    reading the rows of x through the sorted assignments must equal, bit for bit, ops.gather / ops.padded_gather
    (dmoe.py:219 / :273) followed by gmm(trans_a=True), and the CPU oracle's gather and product to 1e-2."""
    torch.manual_seed(tokens + k)
    indices, bin_ids, bins, padded_bins, tpe = _routing(tokens, experts, top_k, seed=tokens + n, blocking=blocking)
    x = torch.randn(tokens, n, device='cuda').to(dtype)
    rows = tokens * top_k if padded_bins is None else int(padded_bins[-1])
    sizes = tpe if padded_bins is None else torch.diff(padded_bins, prepend=padded_bins.new_zeros(1))
    d = torch.randn(rows, k, device='cuda').to(dtype)
    src = gg.GatheredRows(x, indices, bin_ids, bins, padded_bins, top_k, rows)
    guard = torch.full((experts + 2, k, n), 7.0, device='cuda', dtype=dtype)
    got = gg.gmm_tn_gather(d, src, sizes)
    assert got is not None and got.shape == (experts, k, n)
    copy = src.materialize()
    assert torch.equal(got, gg.backend.gmm(d, copy, sizes, trans_a=True))
    again = gg.gmm_tn_gather(d, src, sizes)                       # with the row table the first call left on src
    assert torch.equal(again, got) and getattr(src, '_row_table', None) is not None
    assert torch.equal(src.weight_gradient(d, sizes), got)
    cpu = lambda t: None if t is None else t.cpu()
    if padded_bins is None:
        o_x = oracle.gather(cpu(x), cpu(indices), cpu(bin_ids), None, cpu(bins), top_k)
    else:
        o_x = oracle.padded_gather(cpu(x), cpu(indices), cpu(bin_ids), None, cpu(bins), cpu(padded_bins), top_k)
    want = oracle.gmm(cpu(d), o_x, cpu(sizes), trans_a=True)
    assert rel_err(got.cpu(), want) < TOL
    for e, cnt in enumerate(tpe.tolist()):
        if cnt == 0:
            assert int(torch.count_nonzero(got[e])) == 0          # an expert without tokens: exactly zero
    assert bool((guard == 7.0).all())


def test_gmm_weight_gradient_on_gathered_rows_edge_cases(gg):
    """Assignments outside [0, tokens * top_k) read as rows of zeros; shapes the kernel does not take come back as None
    and `weight_gradient` then gathers once and multiplies."""
    tokens, experts, top_k, n, k = 600, 4, 2, 128, 256
    indices, bin_ids, bins, _, tpe = _routing(tokens, experts, top_k, seed=5)
    x = torch.randn(tokens, n, device='cuda').bfloat16()
    d = torch.randn(tokens * top_k, k, device='cuda').bfloat16()
    bad = indices.clone()
    bad[::7] = -1
    bad[3::11] = tokens * top_k + 5
    got = gg.gmm_tn_gather(d, gg.GatheredRows(x, bad, bin_ids, bins, None, top_k, tokens * top_k), tpe)
    rows_of_x = x[(indices.long() // top_k)].clone()
    rows_of_x[::7] = 0
    rows_of_x[3::11] = 0
    assert torch.equal(got, gg.backend.gmm(d, rows_of_x, tpe, trans_a=True))
    src = gg.GatheredRows(x, indices, bin_ids, bins, None, top_k, tokens * top_k)
    narrow = d[:, :128].contiguous()                               # at most 128 columns: the half-height tile, no gathered form
    assert gg.gmm_tn_gather(narrow, src, tpe) is None
    assert torch.equal(src.weight_gradient(narrow, tpe), gg.backend.gmm(narrow, src.materialize(), tpe, trans_a=True))
    assert gg.gmm_tn_gather(d.float(), gg.GatheredRows(x.float(), indices, bin_ids, bins, None, top_k, tokens * top_k), tpe) is None
    # no tokens at all: every expert's gradient is zero
    none = gg.GatheredRows(x[:0], indices[:0], bin_ids[:0], torch.zeros_like(bins), None, top_k, 0)
    got = gg.gmm_tn_gather(d[:0], none, torch.zeros_like(tpe))
    assert got.shape == (experts, k, n) and not got.any()


def test_gmm_on_gathered_rows_with_assignments_out_of_range(gg):
    """An assignment outside [0, tokens * top_k) reads as a row of zeros (nothing outside x is fetched), and what the
    library has no kernel for comes back as None (the caller gathers first)."""
    tokens, experts, top_k, k, n = 600, 4, 2, 128, 256
    indices, bin_ids, bins, _, tpe = _routing(tokens, experts, top_k, seed=5)
    x = torch.randn(tokens, k, device='cuda').to(torch.bfloat16)
    w1 = (torch.randn(experts, n, k, device='cuda') / k ** 0.5).to(torch.bfloat16)
    bad = indices.clone()
    bad[::7] = -1
    bad[3::11] = tokens * top_k + 5
    src = gg.GatheredRows(x, bad, bin_ids, bins, None, top_k, tokens * top_k)
    (c,) = gg.gmm_gather(src, w1, tpe)
    a = x[(indices.long() // top_k)].clone()
    a[::7] = 0
    a[3::11] = 0
    assert torch.equal(c, gg.backend.gmm(a, w1, tpe, trans_b=True))
    # fp32, a reduction that is not whole K tiles, 64-bit assignments: no kernel
    assert gg.gmm_gather(gg.GatheredRows(x.float(), indices, bin_ids, bins, None, top_k, tokens * top_k), w1.float(), tpe) is None
    assert gg.gmm_gather(gg.GatheredRows(x[:, :72].contiguous(), indices, bin_ids, bins, None, top_k, tokens * top_k),
                         w1[:, :, :72].contiguous(), tpe) is None
    assert gg.gmm_gather(gg.GatheredRows(x, indices.long(), bin_ids, bins, None, top_k, tokens * top_k), w1, tpe) is None


@pytest.mark.parametrize('groups,rows,k,n', [
    (4, 1000, 36, 132),      # K tail of one 16-byte piece, a column tile of one piece
    (3, 65 * 3, 32, 4),      # one K tile, the narrowest output; experts around the 64-row tile
    (8, 8 * 129, 260, 260),  # experts around the full tile
    (1, 300, 2052, 128),     # a handful of tiles, long reduction: cut along K (with and without a workspace)
    (2, 4100, 128, 384),     # TN: few tiles, long reduction
    (70, 2000, 64, 128),     # several experts per lane of the tile lookup, unranked TN
    (5, 40, 128, 4100),      # many column tiles, a few rows per expert
    (60, 12000, 288, 300),   # many small tiles for the columns' sake, a short reduction and a longer one
    (60, 12000, 600, 300),
])
@pytest.mark.parametrize('mode', ['nn', 'nt', 'tn', 'dual_nn', 'dual_nt'])
def test_gmm_fp32_on_the_matrix_cores(gg, monkeypatch, groups, rows, k, n, mode):
    """The fp32 kernels against fp64.  Each of an output's r products and partial sums is rounded once, errors of random
    sign: 2^-24 sqrt(r) relative to the terms' root sum square, with a factor of four to spare."""
    torch.manual_seed(rows + k)
    sizes = _sizes(groups, rows, seed=groups + rows, empty=(0,) if groups > 2 else ())
    trans_b, dual = mode.endswith('nt'), mode.startswith('dual')
    a, a2 = (torch.randn(rows, k, device='cuda') for _ in range(2))
    wshape = (groups, n, k) if trans_b else (groups, k, n)
    b, b2 = (torch.randn(rows, n, device='cuda') if mode == 'tn' else torch.randn(wshape, device='cuda') for _ in range(2))
    # a row that must not leak into its neighbours: the pieces past the end of a row's reduction read as zeros
    bad = rows // 2
    if mode != 'tn':
        a[bad] = float('inf')
    ok = torch.arange(rows, device='cuda') != bad

    def product(x, w):
        outs, start = [], 0
        for e, c in enumerate(sizes.tolist()):
            xe = x[start:start + c].double()
            outs.append(xe.t() @ w[start:start + c].double() if mode == 'tn' else
                        xe @ (w[e].double().t() if trans_b else w[e].double()))
            start += c
        return torch.stack(outs) if mode == 'tn' else torch.cat(outs)

    want = product(a, b) + (product(a2, b2) if dual else 0)
    length = int(sizes.max()) if mode == 'tn' else k * (2 if dual else 1)
    tol = 4 * 2.0 ** -24 * math.sqrt(max(length, 16))
    got = []
    for lend in (True, False):
        monkeypatch.setattr(gg, 'GMM_WORKSPACE', lend)
        for _ in range(2):
            out = gg.gmm_dual(a, b, a2, b2, sizes, trans_b=trans_b) if dual else \
                gg.backend.gmm(a, b, sizes, trans_a=mode == 'tn', trans_b=trans_b)
            if mode == 'tn':
                assert max_block_err(out, want) < tol
            else:
                assert max_block_err(out[ok], want[ok]) < tol and not bool(torch.isfinite(out[bad]).any())
            got.append(out)
        assert torch.equal(got[-1].nan_to_num(), got[-2].nan_to_num())


@pytest.mark.parametrize('mode,rows,k,n', [
    ('nn', 700, 68, 4100), ('nt', 700, 68, 4100), ('dual_nn', 700, 36, 4100), ('dual_nt', 641, 36, 4100),   # 128 x 256
    ('nn', 321, 36, 4100), ('nt', 321, 36, 4100), ('nt', 1300, 68, 260),   # 64 x 128: few rows, few tiles
    ('tn', 700, 260, 4100), ('tn', 700, 132, 4100), ('tn', 700, 132, 260),   # 128 x 256, 256 x 128, 64 x 128
])
def test_gmm_fp32_tiles_with_values_off_the_parts(gg, mode, rows, k, n):
    """Every tile shape of the fp32 kernels, five experts, with rows of the product 2^-100 and 2^45 times the others (tiles formed
    again on the fp32 instruction next to tiles that are not), row by row against fp64: a sum of r terms, with a factor of four to
    spare."""
    torch.manual_seed(rows + k)
    trans_b, dual = mode.endswith('nt'), mode.startswith('dual')
    sizes = _sizes(5, rows, seed=rows)
    wshape = (rows, n) if mode == 'tn' else (5, n, k) if trans_b else (5, k, n)
    a, a2 = (torch.randn(rows, k, device='cuda') for _ in range(2))
    b, b2 = (torch.randn(wshape, device='cuda') for _ in range(2))
    for x in (a, a2):
        view = x.t() if mode == 'tn' else x
        view[3] *= 2.0 ** -100
        view[-2] *= 2.0 ** 45

    def exact(x, w):
        parts = list(zip(x.double().split(sizes.tolist()), w.double().split(sizes.tolist()) if mode == 'tn' else w.double()))
        return torch.cat([p.t() @ q if mode == 'tn' else p @ (q.t() if trans_b else q) for p, q in parts])
    want = exact(a, b) + (exact(a2, b2) if dual else 0)
    got = gg.gmm_dual(a, b, a2, b2, sizes, trans_b=trans_b) if dual else gg.backend.gmm(a, b, sizes, trans_a=mode == 'tn', trans_b=trans_b)
    got = got.double().reshape(want.shape)
    length = int(sizes.max()) if mode == 'tn' else k * (2 if dual else 1)
    error = (got - want).norm(dim=1) / want.norm(dim=1).clamp_min(1e-300)
    assert float(error.max()) < 4 * 2.0 ** -24 * math.sqrt(max(length, 16)), error.argmax()


@pytest.mark.parametrize('other', [float('inf'), float('nan'), 2.0 ** 40, 2.0 ** -80])
@pytest.mark.parametrize('mode', ['nn', 'nt', 'dual_nn', 'dual_nt'])
def test_gmm_fp32_rows_do_not_depend_on_the_rows_behind_them(gg, mode, other):
    """An expert's rows give the same bits whatever the next expert's rows, and rows behind the last bin, hold: a row tile
    reaches past the rows it belongs to (70 and 200 rows; tiles of 64 and 128)."""
    torch.manual_seed(3)
    k, n, trans_b, dual = 512, 260, mode.endswith('nt'), mode.startswith('dual')
    for first, second, behind in ((70, 50, 40), (400, 300, 100)):
        a, a2 = (torch.randn(first + second + behind, k, device='cuda') for _ in range(2))
        b, b2 = (torch.randn((2, n, k) if trans_b else (2, k, n), device='cuda') for _ in range(2))
        sizes = torch.tensor([first, second], device='cuda')     # on the device: their sum need not be the row count

        def product(x, x2):
            return gg.gmm_dual(x, b, x2, b2, sizes, trans_b=trans_b) if dual else gg.backend.gmm(x, b, sizes, trans_b=trans_b)
        want = product(a, a2)[:first + second]
        x, x2 = a.clone(), a2.clone()
        x[first + second:], x2[first + second:] = other, other
        assert torch.equal(product(x, x2)[:first + second], want)
        x[first:], x2[first:] = other, other
        assert torch.equal(product(x, x2)[:first], want[:first])


@pytest.mark.parametrize('k', [36, 64, 2052])
@pytest.mark.parametrize('mode', ['nn', 'nt', 'tn'])
def test_gmm_fp32_at_the_ends_of_the_range(gg, k, mode):
    """Output rows from operands next to the largest and the smallest fp32 values, which are not the sum of three bf16 values
    there, against fp64.  Every row is held to the error of a sum of k terms, 2^-24 sqrt(k) of its largest entry with a
    factor of four to spare, plus what underflow leaves of a product."""
    torch.manual_seed(k)
    rows, n = 300, 132
    a = torch.randn(rows, k, device='cuda')
    b = torch.randn(k, n, device='cuda').clamp_(-3, 3)
    a *= torch.exp2(-torch.arange(rows, device='cuda').float() / 2.25).unsqueeze(1)   # down to 2^-133: subnormals
    a[7], a[8], a[9] = 0.0, 0.0, 0.0
    largest = torch.finfo(torch.float32).max
    a[7, 3], a[8, k - 1], a[200, k // 2] = largest, -largest, largest
    b[3], b[k - 1], b[k // 2] = b[3] / 4, b[k - 1] / 4, b[k // 2] / 4
    want = a.double() @ b.double()
    sizes = torch.tensor([rows])
    if mode == 'tn':
        got = gg.backend.gmm(a.t().contiguous(), b, torch.tensor([k]), trans_a=True)[0]
    else:
        got = gg.backend.gmm(a, (b.t() if mode == 'nt' else b).contiguous()[None], sizes, trans_b=mode == 'nt')
    tol = 4 * 2.0 ** -24 * math.sqrt(k) * want.abs().amax(1) + k * 2.0 ** -149
    assert bool(((got.double() - want).abs().amax(1) <= tol).all())
    assert not bool(got[9].any())


@pytest.mark.parametrize('r', [124, 160, 700])   # 700: cut reductions
@pytest.mark.parametrize('mode', ['nn', 'nt', 'tn', 'dual_nn', 'dual_nt'])
def test_gmm_fp32_every_sum_has_the_bits_of_its_own_terms(gg, mode, r):
    """Operands whose large values meet zeros or small ones of the other, so that a sum is made of values far below the largest of its row and
    column.  First rows of either operand with zeros, a late value 2^10 or 2^30 times as large, later values 2^-12 or 2^-40 of the first, one value
    only; a NaN, an infinity.  Then every k of one operand times 2^u, u in -16 .. 16, and of the other times 2^-u.  Every sum by itself against
    fp64, over the sum of its terms' magnitudes: three bf16 parts a value leave out up to 2.6 2^-24 of a term, an accumulator is rounded six times
    per 32 terms, 2^-25 of what it holds each, of which the root counts (errors of either sign), with a factor of two to spare.  Not finite is
    what is in the row of a NaN or an infinity, and nothing else."""
    torch.manual_seed(r)
    rows, n, trans_b, dual = 152, 260, mode.endswith('nt'), mode.startswith('dual')

    def operand(count):     # [count, r]: a row of it is one reduction
        x = torch.randn(count, r, device='cuda')
        x[1, :64] = 0
        x[2, r - 1], x[3, r - 1] = 2.0 ** 10, 2.0 ** 30
        x[4, 64:] *= 2.0 ** -12
        x[5, 64:] *= 2.0 ** -40
        x[6] = 0
        x[6, r - 3] = 2.0 ** -90
        x[7, :] = 0
        x[8] *= 2.0 ** 60
        return x

    def product(x, w, x2, w2):
        if mode == 'tn':
            return gg.backend.gmm(x.t().contiguous(), w.t().contiguous(), torch.tensor([r]), trans_a=True)[0]
        w, w2 = ((v if trans_b else v.t().contiguous())[None] for v in (w, w2))
        sizes = torch.tensor([rows])
        return gg.gmm_dual(x, w, x2, w2, sizes, trans_b=trans_b) if dual else gg.backend.gmm(x, w, sizes, trans_b=trans_b)

    def against_fp64(a, b, a2, b2):
        want, terms = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
        if dual:
            want, terms = want + a2.double() @ b2.double().t(), terms + a2.double().abs() @ b2.double().abs().t()
        return want, terms + 2.0 ** -110   # fp32 resolves 2^-149 at the smallest

    tol = 2.0 ** -24 * 2 * (2.6 + math.sqrt(6 * (2 * r if dual else r) / 32) / 2)
    a, b, a2, b2 = operand(rows), operand(n), operand(rows), operand(n)
    want, terms = against_fp64(a, b, a2, b2)
    got = product(a, b, a2, b2).double()
    assert float(((got - want).abs() / terms).max()) < tol
    assert bool((got[7] == 0).all()) and bool((got[:, 7] == 0).all())
    rest = torch.arange(rows, device='cuda') != 40
    for value, at in ((float('nan'), r // 2), (float('inf'), r - 1)):
        x = a.clone()
        x[40, at] = value
        got = product(x, b, a2, b2).double()
        assert not bool(torch.isfinite(got[40, torch.arange(n, device='cuda') != 7]).any())
        assert float(((got - want).abs() / terms)[rest].max()) < tol
    a, b, a2, b2 = (torch.randn(count, r, device='cuda') for count in (rows, n, rows, n))
    up, up2 = (2.0 ** torch.randint(-16, 17, (r,), device='cuda').float() for _ in range(2))
    a, b, a2, b2 = a * up, b / up, a2 * up2, b2 / up2
    want, terms = against_fp64(a, b, a2, b2)
    assert float(((product(a, b, a2, b2).double() - want).abs() / terms).max()) < tol


@pytest.mark.parametrize('dtype,mode', [(torch.float32, 'nn'), (torch.float32, 'nt'), (torch.float32, 'tn'), (torch.bfloat16, 'nn')])
def test_captures_have_workspaces_of_their_own(gg, dtype, mode):
    """Two graphs captured one after the other on one stream, with products whose tiles are cut along the reduction: replayed
    in either order, next to eager products, each gives the eager result bit for bit."""
    torch.manual_seed(3)
    groups, rows, k, n = 1, 256, 4096, 512
    if mode == 'tn':
        a, b, sizes = torch.randn(k, rows, device='cuda').to(dtype), torch.randn(k, n, device='cuda').to(dtype), [k]
    else:
        a = torch.randn(rows, k, device='cuda').to(dtype)
        b, sizes = torch.randn(groups, *((n, k) if mode == 'nt' else (k, n)), device='cuda').to(dtype), [rows]
    sizes = torch.tensor(sizes, device='cuda')

    def product():
        return gg.backend.gmm(a, b, sizes, trans_a=mode == 'tn', trans_b=mode == 'nt')

    want = product()
    torch.cuda.synchronize()
    graphs, outs, used = [], [], [gg._workspace(a.device)[0]]
    for _ in range(2):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outs.append((product(), product()))
            used.append(gg._workspace(a.device)[0])
            assert gg._workspace(a.device)[0] == used[-1]
        graphs.append(graph)
    assert len(set(used)) == 3
    for order in ((1, 0), (0, 1), (1, 1, 0)):
        for i in order:
            for out in outs[i]:
                out.zero_()
            graphs[i].replay()
            eager = product()
            torch.cuda.synchronize()
            assert all(torch.equal(out, want) for out in (*outs[i], eager))


@pytest.mark.parametrize('among', [0, 64, 300])
def test_gmm_fp32_of_few_terms(gg, among):
    """Weight gradients of experts with one to eight rows, by themselves and next to experts of `among` rows on average: the error
    against fp64 is no larger than that of a chain of fp32 multiply-adds (one term: the product, rounded once)."""
    torch.manual_seed(among)
    k, n, terms = 260, 516, list(range(1, 9))
    sizes = torch.tensor(terms + ([16 * among - 4] if among else []))
    rows = int(sizes.sum())
    a, b = torch.randn(rows, k, device='cuda'), torch.randn(rows, n, device='cuda')
    out = gg.backend.gmm(a, b, sizes, trans_a=True)
    start = 0
    for e, r in enumerate(terms):
        x, y = a[start:start + r].double(), b[start:start + r].double()
        start += r
        want, chain = x.t() @ y, torch.zeros(k, n, device='cuda')
        for t in range(r):
            chain = (chain.double() + x[t, :, None] * y[t, None, :]).float()   # exact product, one rounding
        if r == 1:
            assert torch.equal(out[e], chain)
        total = x.abs().t() @ y.abs()
        for norm in (lambda d: float(d.norm()), lambda d: float((d / total).abs().max())):
            assert norm(out[e].double() - want) <= 1.05 * norm(chain.double() - want), (r, norm(out[e].double() - want), norm(chain.double() - want))


@pytest.mark.parametrize('small,large', [(-128, 20), (-136, 30), (-149, 37), (-140, 100)])
@pytest.mark.parametrize('mode', ['nn', 'nt', 'tn', 'dual_nn', 'dual_nt'])
def test_gmm_fp32_of_values_without_bf16_parts(gg, mode, small, large):
    """Values below the smallest bf16 value, whose three parts are all zero, times large ones, in either operand, among rows
    of zeros: the sums, far inside the fp32 range, come out of the values themselves.  Bound of a sum of k terms, with a
    factor of four to spare."""
    torch.manual_seed(-small)
    rows, k, n, trans_b, dual = 200, 68, 132, mode.endswith('nt'), mode.startswith('dual')
    tiny = (torch.rand(rows, k, device='cuda', dtype=torch.float64) + 1) * 2.0 ** small
    tiny = tiny.float()
    tiny[rows // 2:rows // 2 + 20] = 0
    big = (torch.rand(rows, n, device='cuda') + 1) * 2.0 ** large if mode == 'tn' else (torch.rand(1, k, n, device='cuda') + 1) * 2.0 ** large
    sizes = torch.tensor([rows])
    tol = 4 * 2.0 ** -24 * math.sqrt(2 * (rows if mode == 'tn' else k))

    def product(x, w):
        if mode == 'tn':
            return gg.backend.gmm(x, w, sizes, trans_a=True)[0]
        w = w.transpose(1, 2).contiguous() if trans_b else w
        return gg.gmm_dual(x, w, x, w, sizes, trans_b=trans_b) if dual else gg.backend.gmm(x, w, sizes, trans_b=trans_b)

    def exact(x, w):
        return x.double().t() @ w.double() if mode == 'tn' else (2 if dual else 1) * (x.double() @ w[0].double())

    def check(x, w):
        want, got = exact(x, w), product(x, w).double()
        assert float((got - want).norm() / want.norm()) < tol + 2.0 ** -149 / float(want.abs().max())
        assert bool((got[want == 0] == 0).all())
    check(tiny, big)
    if mode == 'tn':
        check(big, tiny)
    else:   # the other way round: rows of large values, tiny weights
        check((torch.rand(rows, k, device='cuda') + 1) * 2.0 ** large, (tiny[:k, :1].expand(k, n) * 1.0).unsqueeze(0).contiguous())
    # next to values of ordinary size in the same tile, a row and a column of them
    x, w = torch.randn_like(tiny), big.clone()
    if mode != 'tn':
        x[3] = tiny[3]
        got, want = product(x, w).double(), exact(x, w)
        assert float((got[3] - want[3]).norm() / want[3].norm()) < tol


@pytest.mark.parametrize('power', [37, 110, 126])
@pytest.mark.parametrize('mode', ['nn', 'nt', 'tn'])
def test_gmm_fp32_of_small_by_large_values(gg, mode, power):
    """Values around 2^-power times values around 2^power, sums around 1, against fp64: the small ones have parts below the
    normal range of bf16 from about 2^-102 on.  The error bound of a sum of k terms, with a factor of four to spare."""
    torch.manual_seed(power)
    rows, k, n = 200, 96, 132
    a = torch.randn(rows, k, device='cuda').clamp_(-3, 3) * 2.0 ** -power
    b = torch.randn(k, n, device='cuda').clamp_(-1.9, 1.9) * 2.0 ** power
    want = a.double() @ b.double()
    if mode == 'tn':
        got = gg.backend.gmm(a.t().contiguous(), b, torch.tensor([k]), trans_a=True)[0]
    else:
        got = gg.backend.gmm(a, (b.t() if mode == 'nt' else b).contiguous()[None], torch.tensor([rows]), trans_b=mode == 'nt')
    assert max_block_err(got, want) < 4 * 2.0 ** -24 * math.sqrt(k)


@pytest.mark.parametrize('groups,rows,k,n', [(3, 700, 8, 136), (4, 900, 72, 264), (5, 1500, 200, 512), (8, 3000, 1032, 2728),
                                             (2, 40, 312, 1032), (12, 3600, 2728, 1032), (1, 260, 4104, 64)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_gmm_reductions_that_end_inside_a_k_tile(gg, monkeypatch, groups, rows, k, n, dtype):
    """k a multiple of 8 but not of 64, every NN / NT form, against fp32.  One row of the first operand and one weight row
    are infinite: nothing of them may reach the products of the rows in front of them, whose last pieces end where
    these begin in memory."""
    torch.manual_seed(k)
    sizes = _sizes(groups, rows, seed=k + rows, empty=(0,) if groups > 2 else ())
    a, a2 = (torch.randn(rows, k, device='cuda').to(dtype) for _ in range(2))
    wt, wt2 = ((torch.randn(groups, n, k, device='cuda') / k ** 0.5).to(dtype) for _ in range(2))      # NT
    w, w2 = ((torch.randn(groups, k, n, device='cuda') / k ** 0.5).to(dtype) for _ in range(2))        # NN
    bad_row, bad_col = rows // 2, n - 1
    a[bad_row] = float('inf')
    wt[:, bad_col] = float('inf')
    keep = torch.ones(rows, n, dtype=torch.bool, device='cuda')
    keep[bad_row] = False
    nt_keep = keep.clone()
    nt_keep[:, bad_col] = False

    def check(got, want, mask):
        got, want = (torch.where(mask, t.float(), torch.zeros((), device='cuda')) for t in (got, want))
        assert max_block_err(got, want) < TOL

    nt, nn = _ref_gpu(a, wt, sizes, False, True), _ref_gpu(a, w, sizes, False, False)
    nt2, nn2 = _ref_gpu(a2, wt2, sizes, False, True), _ref_gpu(a2, w2, sizes, False, False)
    for lend in (True, False):
        monkeypatch.setattr(gg, 'GMM_WORKSPACE', lend)
        check(gg.backend.gmm(a, wt, sizes, trans_b=True), nt, nt_keep)
        check(gg.backend.gmm(a, w, sizes), nn, keep)
        check(gg.gmm_dual(a, wt, a2, wt2, sizes, trans_b=True), nt + nt2, nt_keep)
        check(gg.gmm_dual(a, w, a2, w2, sizes), nn + nn2, keep)
    gelu = lambda t: torch.nn.functional.gelu(t.to(dtype).float(), approximate='tanh')   # noqa: E731
    pre, act = gg.gmm_act(a, wt, sizes, fuse=True)
    check(pre, nt, nt_keep)
    check(act, gelu(pre), nt_keep)
    x1, x2, h = gg.gmm_glu(a, wt, wt2, sizes, 1, fuse=True)
    x2_ref = _ref_gpu(a, wt2, sizes, False, True)
    check(x1, nt, nt_keep)
    check(x2, x2_ref, keep)
    check(h, gelu(x1) * x2.float(), nt_keep)
    saved, saved2 = (torch.randn(rows, n, device='cuda').to(dtype) for _ in range(2))
    check(gg.gmm_dact(a, wt, saved, sizes, fuse=True), gg.gmm_dact(a, wt, saved, sizes, fuse=False), nt_keep)
    for got, want in zip(gg.gmm_dglu(a, wt, saved, saved2, sizes, 0, fuse=True), gg.gmm_dglu(a, wt, saved, saved2, sizes, 0, fuse=False)):
        check(got, want, nt_keep)
    # the combine in the store phase
    order = torch.randperm(rows, device='cuda').int()
    bins = torch.cumsum(sizes.cuda(), 0).int()
    bin_ids = torch.repeat_interleave(torch.arange(groups), sizes).int().cuda()
    weights = torch.rand(rows, device='cuda').to(dtype)
    y, out = gg.gmm_scatter(a, w, sizes, gg.CombinedRows(order, bin_ids, bins, weights))
    check(y, nn, keep)
    want = torch.zeros_like(out)
    want[order.long()] = (y.float() * weights[order.long()].float()[:, None]).to(dtype)
    placed = torch.ones_like(keep)
    placed[order[bad_row].long()] = False
    assert torch.equal(torch.where(placed, out, 0), torch.where(placed, want, 0))


@pytest.fixture
def row_kernel():
    """Names the kernel that takes this thread's NN / NT products: 1 the general one, 2 that of launches of few tiles (an error
    where it cannot)."""
    from megablocks_amd._lib import lib
    yield lib.mbx_debug_row_kernel
    lib.mbx_debug_row_kernel(0)


@pytest.mark.parametrize('counts,k,n', [
    ([100, 0, 129, 128, 1, 300], 128, 136), ([257, 255, 64], 200, 520), ([200], 64, 8), ([90] * 16, 448, 1032), ([60, 500], 8, 264),
    ([61] * 70, 64, 72),
    ([1], 8, 8), ([127, 1, 0, 128], 72, 128), ([300, 290, 310], 2728, 1032), ([1, 2, 3], 576, 2048)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_products_of_few_tiles_are_the_general_kernels(gg, monkeypatch, row_kernel, counts, k, n, dtype):
    """Launches of few tiles have a kernel of their own, every form of which gives the bits of the general one's: each is run by
    both, at reductions that end inside a K tile, rows and columns inside a tile, more experts than a wave has lanes and operands
    with rows behind the last expert's; the plain products also against fp32."""
    torch.manual_seed(k + n)
    monkeypatch.setattr(gg, 'GMM_WORKSPACE', False)   # no cut along the reduction
    sizes = torch.tensor(counts, device='cuda')       # on the device: their sum need not be the row count
    groups, rows = len(counts), sum(counts)
    m = rows + 37
    a, a2, p1, p2 = ((torch.randn(m, w, device='cuda')).to(dtype) for w in (k, k, n, n))
    wt, wt2 = ((torch.randn(groups, n, k, device='cuda') / k ** 0.5).to(dtype) for _ in range(2))
    w, w2 = (t.transpose(1, 2).contiguous() for t in (wt, wt2))
    order = torch.randperm(rows, device='cuda').int()
    bins = torch.cumsum(sizes, 0).int()
    bin_ids = torch.repeat_interleave(torch.arange(groups, device='cuda'), sizes).int()
    weights = torch.rand(m, device='cuda').to(dtype)
    tokens = torch.randn(rows, k, device='cuda').to(dtype)

    def forms():
        src = gg.GatheredRows(tokens, order, bin_ids, bins, None, 1, m)
        out = [gg.backend.gmm(a, wt, sizes, trans_b=True), gg.backend.gmm(a, w, sizes), gg.gmm_dact(a, wt, p1, sizes, fuse=True)]
        if k > 192:
            out += [gg.gmm_dual(a, wt, a2, wt2, sizes, trans_b=True), gg.gmm_dual(a, w, a2, w2, sizes)]
        out += [*gg.gmm_act(a, wt, sizes, fuse=True), *gg.gmm_act(a, w, sizes, fuse=True, trans_b=False)]
        for act in (0, 1):
            out += [*gg.gmm_glu(a, wt, wt2, sizes, act, fuse=True), *gg.gmm_dglu(a, wt, p1, p2, sizes, act, fuse=True)]
        if k % 64 == 0:
            for act, second in ((None, None), (1, None), (0, wt2), (1, wt2)):
                out += [*gg.gmm_gather(src, wt, sizes, act=act, b2=second)]
                if act is not None:
                    out += [gg.gmm_gather(src, wt, sizes, act=act, b2=second, keep_product=False)[-1]]
        combine = gg.CombinedRows(torch.cat([order, torch.zeros(m - rows, dtype=torch.int32, device='cuda')]), bin_ids, bins, weights)
        y, combined = gg.gmm_scatter(a, w, sizes, combine)
        return [t[:rows] for t in out + [y] if t is not None], combined[order.long()]
    row_kernel(1)
    general, placed = forms()
    assert row_kernel(2) == 1
    here, placed_here = forms()
    assert row_kernel(0) == 2
    assert len(here) == len(general) and all(torch.equal(s, t) for s, t in zip(here, general))
    assert torch.equal(placed, placed_here)
    for layout, got in ((True, here[0]), (False, here[1])):
        want = _ref_gpu(a[:rows], wt if layout else w, sizes.cpu(), False, layout)
        assert max_block_err(got, want) < TOL


@pytest.mark.parametrize('counts,k,n', [
    ([100, 0, 128, 60], 4096, 520),            # no full round, half-height tiles: eight parts
    ([700, 20, 300], 4104, 264),               # full tiles, a reduction that ends inside a K tile
    ([250, 270] * 32, 4096, 1024),             # behind two rounds of half-height tiles: two parts
    ([250, 270] * 32, 2048, 1024),             # ... of too few K tiles: not cut
    ([1024] * 8, 5184, 2304),                  # behind a full round: eight parts
    ([1024] * 8, 2048, 2304),                  # ... where half-height tiles are shorter: not cut
])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_combine_in_the_store_phase_of_tiles_cut_along_the_reduction(gg, monkeypatch, row_kernel, counts, k, n, dtype):
    """Product and combined output, with and without the product kept, are those of the cut product and the combine after it, bit for
    bit, on the last of three launches too, which find the counters as the first did."""
    torch.manual_seed(k + n)
    sizes = torch.tensor(counts)
    groups, rows = len(counts), int(sizes.sum())
    a = torch.randn(rows, k, device='cuda').to(dtype)
    w = (torch.randn(groups, k, n, device='cuda') / k ** 0.5).to(dtype)
    order = torch.randperm(rows, device='cuda').int()
    bins = torch.cumsum(sizes.cuda(), 0).int()
    bin_ids = torch.repeat_interleave(torch.arange(groups), sizes).int().cuda()
    combine = gg.CombinedRows(order, bin_ids, bins, torch.rand(rows, device='cuda').to(dtype))
    row_kernel(1)
    y = gg.backend.gmm(a, w, sizes)
    want = combine.scatter(y)
    for keep in (True, False, True):
        got, out = gg.gmm_scatter(a, w, sizes, combine, keep_product=keep)
        assert torch.equal(out, want) and (torch.equal(got, y) if keep else got is None)
    monkeypatch.setattr(gg, 'GMM_WORKSPACE', False)
    whole, out = gg.gmm_scatter(a, w, sizes, combine)
    assert torch.equal(whole, y) == (k == 2048)   # the other launches were cut
    assert rel_err(y, whole) < TOL and rel_err(want, out) < TOL


@pytest.mark.parametrize('combined', [False, True])
def test_tiles_cut_along_the_reduction_are_the_same_every_time(gg, row_kernel, combined):
    """The workgroup that comes last puts the sum of the parts where the count of the parts was: every one of many launches gives the same
    bits and leaves the counters at zero.  32 tiles of eight parts fill the chip with such hand-overs."""
    from megablocks_amd import _lib
    torch.manual_seed(5)
    sizes, k, n = torch.tensor([1000, 1024]), 4096, 1024
    a = torch.randn(2024, k, device='cuda').bfloat16()
    w = (torch.randn(2, k, n, device='cuda') / k ** 0.5).bfloat16()
    bins = torch.cumsum(sizes.cuda(), 0).int()
    bin_ids = torch.repeat_interleave(torch.arange(2), sizes).int().cuda()
    combine = gg.CombinedRows(torch.randperm(2024, device='cuda').int(), bin_ids, bins, torch.rand(2024, device='cuda').bfloat16())
    row_kernel(1)
    run = (lambda: gg.gmm_scatter(a, w, sizes, combine)[1]) if combined else (lambda: gg.backend.gmm(a, w, sizes))
    first = run()
    y = gg.backend.gmm(a, w, sizes)
    assert max_block_err(y, _ref_gpu(a, w, sizes, False, False)) < 2 * TOL
    assert torch.equal(first, combine.scatter(y) if combined else y)
    different = sum((run() != first).any().int() for _ in range(100))
    assert int(different) == 0
    ws = gg._workspaces[(torch.cuda.current_device(), _lib.stream().value)]
    assert int(ws[:4096].count_nonzero()) == 0


@pytest.mark.parametrize('counts,k,n', [
    ([0, 1, 16, 17, 33, 2, 0, 0, 3, 5, 1, 0], 2048, 136),      # experts around the 16 rows a workgroup takes
    ([1] + [0] * 7, 4096, 1024), ([3, 0, 0, 1] + [0] * 60, 2048, 1408), ([2] * 16, 200, 264), ([1, 2, 1, 4] * 20, 2728, 72),
    ([5] * 8, 64, 64), ([8] * 3, 8, 8),
])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_gmm_with_a_handful_of_rows_per_expert(gg, counts, k, n, dtype):
    """The kernels for a few rows per expert, every form they take, against fp32; k also inside a chunk, where a row's last
    piece ends in front of a row of infinities; the forms' products equal bit for bit, and from run to run."""
    torch.manual_seed(k + n)
    sizes = torch.tensor(counts)
    groups, rows = len(counts), int(sizes.sum())
    a = torch.randn(rows, k, device='cuda').to(dtype)
    w1, v1 = ((torch.randn(groups, n, k, device='cuda') / k ** 0.5).to(dtype) for _ in range(2))
    w2 = (torch.randn(groups, k, n, device='cuda') / k ** 0.5).to(dtype)
    bad = rows // 2
    w1[:, n - 1] = float('inf')
    keep = torch.ones(rows, n, dtype=torch.bool, device='cuda')
    if rows > 1:
        a[bad] = float('inf')
        keep[bad] = False
    nt_keep = keep.clone()
    nt_keep[:, n - 1] = False

    def check(got, want, mask):
        got, want = (torch.where(mask, t.float(), torch.zeros((), device='cuda')) for t in (got, want))
        assert rel_err(got, want) < TOL and max_block_err(got, want, 8, 32) < 4 * TOL

    c = gg.backend.gmm(a, w1, sizes, trans_b=True)
    check(c, _ref_gpu(a, w1, sizes, False, True), nt_keep)
    assert torch.equal(c[:, :n - 1][keep[:, :n - 1]], gg.backend.gmm(a, w1, sizes, trans_b=True)[:, :n - 1][keep[:, :n - 1]])
    finite = lambda t: torch.where(nt_keep, t, torch.zeros((), dtype=dtype, device='cuda'))   # noqa: E731
    pre, act = gg.gmm_act(a, w1, sizes, fuse=True)
    assert torch.equal(finite(pre), finite(c))
    check(act, torch.nn.functional.gelu(c.float(), approximate='tanh'), nt_keep)
    for code, fn in ((0, torch.nn.functional.silu), (1, lambda t: torch.nn.functional.gelu(t, approximate='tanh'))):
        x1, x2, h = gg.gmm_glu(a, w1, v1, sizes, code, fuse=True)
        assert torch.equal(finite(x1), finite(c))
        check(x2, _ref_gpu(a, v1, sizes, False, True), keep)
        check(h, fn(x1.float()).to(dtype).float() * x2.float(), nt_keep)
    y = gg.backend.gmm(a, w2, sizes)
    check(y, _ref_gpu(a, w2, sizes, False, False), keep)
    # one expert per token: the rows picked from, and combined to, the tokens' places
    order = torch.randperm(rows, device='cuda').int()
    bins = torch.cumsum(sizes.cuda(), 0).int()
    bin_ids = torch.repeat_interleave(torch.arange(groups), sizes).int().cuda()
    weights = torch.rand(rows, device='cuda').to(dtype)
    y2, out = gg.gmm_scatter(a, w2, sizes, gg.CombinedRows(order, bin_ids, bins, weights))
    assert torch.equal(y2[keep], y[keep])
    placed = torch.ones(rows, dtype=torch.bool, device='cuda')
    placed[order[bad].long()] = rows == 1
    want = gg.CombinedRows(order, bin_ids, bins, weights).scatter(y)
    assert torch.equal(out[placed], want[placed])
    if k % 64 == 0:
        src = gg.GatheredRows(a, order, bin_ids, bins, None, 1, rows)
        (g,) = gg.gmm_gather(src, w1, sizes)
        mask = keep[order.long()] & nt_keep[0]
        assert torch.equal(g[mask], gg.backend.gmm(src.materialize(), w1, sizes, trans_b=True)[mask])


@pytest.mark.parametrize('counts,k,n', [
    ([33, 1, 0, 70, 2, 0, 0, 1, 0, 0, 0, 0, 0, 0, 17, 4], 2048, 1096),      # columns that end inside a run of eight tiles
    ([0] * 15 + [128], 2048, 512), ([0, 64] + [0] * 30, 2056, 72), ([7] * 8, 2816, 8448), ([56] + [0] * 7, 4096, 1032),
    ([4] * 12, 3072, 4096), ([8, 8], 3072, 264),
])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_gmm_with_a_handful_of_rows_on_average(gg, counts, k, n, dtype):
    """The same where single experts have several row tiles of those kernels, and on both sides of the lines to the others."""
    test_gmm_with_a_handful_of_rows_per_expert(gg, counts, k, n, dtype)


@pytest.mark.parametrize('counts,k,n', [
    ([2] * 16, 4096, 1032), ([1, 0, 5, 4] * 8, 2048, 520), ([8] * 6, 200, 136),      # a handful of rows per expert
    ([17, 24, 40] * 11, 264, 2056), ([130, 90, 200, 64], 136, 776), ([300] * 8, 1088, 264),
])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_products_under_an_epilogue_are_the_plain_ones(gg, monkeypatch, counts, k, n, dtype):
    """Every epilogue is applied to the product the plain launch forms, bit for bit, whichever kernel takes the sizes:
    with activations where the derivative is 1 (gelu_tanh and SiLU far to the right) the gradient forms show it too."""
    torch.manual_seed(n)
    monkeypatch.setattr(gg, 'GMM_WORKSPACE', False)      # lent memory would let plain NN launches cut their last tiles
    sizes = torch.tensor(counts)
    groups, rows = len(counts), int(sizes.sum())
    sizes = sizes.cuda()
    a = torch.randn(rows, k, device='cuda').to(dtype)
    w, v = ((torch.randn(groups, n, k, device='cuda') / k ** 0.5).to(dtype) for _ in range(2))
    plain, plain_v = gg.backend.gmm(a, w, sizes, trans_b=True), gg.backend.gmm(a, v, sizes, trans_b=True)
    right = torch.full((rows, n), 32.0, device='cuda', dtype=dtype)
    assert torch.equal(gg.gmm_act(a, w, sizes, fuse=True)[0], plain)
    assert torch.equal(gg.gmm_dact(a, w, right, sizes, fuse=True), plain)
    for code in (0, 1):
        x1, x2, _ = gg.gmm_glu(a, w, v, sizes, code, fuse=True)
        assert torch.equal(x1, plain) and torch.equal(x2, plain_v)
        d1, d2 = gg.gmm_dglu(a, w, right, torch.full_like(right, 0.5), sizes, code, fuse=True)
        assert torch.equal(d1, plain * 0.5) and torch.equal(d2, plain * 32)
    wn = w.transpose(1, 2).contiguous()
    nn = gg.backend.gmm(a, wn, sizes)
    pre, act = gg.gmm_act(a, wn, sizes, fuse=True, trans_b=False)
    assert torch.equal(pre, nn)
    assert rel_err(act, torch.nn.functional.gelu(pre.float(), approximate='tanh')) < 4e-3     # one rounding step
    order = torch.arange(rows, device='cuda').int()
    bin_ids = torch.repeat_interleave(torch.arange(groups, device='cuda'), sizes).int()
    y, _ = gg.gmm_scatter(a, wn, sizes, gg.CombinedRows(order, bin_ids, torch.cumsum(sizes, 0).int(), None))
    assert torch.equal(y, nn)


@pytest.mark.parametrize('groups,rows,k,n', [(1, 1, 8, 8), (3, 130, 64, 256), (5, 1280, 72, 264), (8, 8 * 257, 128, 1032), (32, 4096, 192, 768)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_batched_mlp_with_activation_epilogues(gg, monkeypatch, groups, rows, k, n, dtype):
    """The capacity-factor layer's products with the activation in their epilogues against the plain product and an
    element-wise pass: the product bit for bit unless the plain launch cuts its last tiles along the reduction, the
    activation of the stored product within the rounding of two tanh evaluations; and every gradient against the node
    autograd builds from the parts."""
    from megablocks_amd.layers.mlp import BatchedGeluMLP
    torch.manual_seed(rows)
    sizes = _sizes(groups, rows, seed=rows, empty=(1,) if groups > 2 else ()).cuda()
    x = torch.randn(rows, k, device='cuda').to(dtype)
    w1 = (torch.randn(groups, k, n, device='cuda') / k ** 0.5).to(dtype)
    w2 = (torch.randn(groups, n, k, device='cuda') / n ** 0.5).to(dtype)
    pre, act = gg.gmm_act(x, w1, sizes, fuse=True, trans_b=False)
    assert max_block_err(pre, _ref_gpu(x, w1, sizes.cpu(), False, False)) < TOL
    assert rel_err(act, torch.nn.functional.gelu(pre.float(), approximate='tanh')) < TOL
    monkeypatch.setattr(gg, 'GMM_WORKSPACE', False)
    assert torch.equal(pre, gg.backend.gmm(x, w1, sizes))
    monkeypatch.undo()
    grad = torch.randn(rows, k, device='cuda').to(dtype)
    results = []
    for fused in (True, False):
        ts = [t.clone().requires_grad_(True) for t in (x, w1, w2)]
        if fused:
            y = BatchedGeluMLP.apply(*ts, sizes)
        else:
            h = torch.nn.functional.gelu(gg.ops.gmm(ts[0], ts[1], sizes), approximate='tanh')
            y = gg.ops.gmm(h, ts[2], sizes)
        y.backward(grad)
        results.append([y] + [t.grad for t in ts])
    for got, want in zip(*results):
        assert rel_err(got, want) < TOL
    # inputs without a gradient: nothing is computed for them
    w = w2.clone().requires_grad_(True)
    BatchedGeluMLP.apply(x, w1, w, sizes).backward(grad)
    assert torch.equal(w.grad, results[0][3])


@pytest.mark.parametrize('groups,tokens,top_k,k,n', [(1, 1, 1, 64, 8), (4, 30, 2, 128, 264), (3, 130, 1, 72, 256), (8, 700, 2, 64, 1032),
                                                     (5, 2000, 3, 128, 136), (2, 900, 2, 192, 512)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_first_products_that_write_only_their_activation(gg, groups, tokens, top_k, k, n, dtype):
    """Without gradients the launches leave the products themselves out: the activation bit for bit, for every form."""
    torch.manual_seed(tokens)
    rows = tokens * top_k
    sizes = _sizes(groups, rows, seed=rows, empty=(0,) if groups > 2 else ()).cuda()
    x = torch.randn(tokens, k, device='cuda').to(dtype)
    b1, b2 = ((torch.randn(groups, n, k, device='cuda') / k ** 0.5).to(dtype) for _ in range(2))
    order = torch.randperm(rows, device='cuda').int()
    bins = torch.cumsum(sizes, 0).int()
    bin_ids = torch.repeat_interleave(torch.arange(groups, device='cuda'), sizes.long()).int()
    padded_sizes = ((sizes + 127) // 128 * 128).int()
    padded = torch.cumsum(padded_sizes, 0).int()
    for src, group_sizes in ((gg.GatheredRows(x, order, bin_ids, bins, None, top_k, rows), sizes),
                             (gg.GatheredRows(x, order, bin_ids, bins, padded, top_k, int(padded[-1])), padded_sizes)):
        a = src.materialize()
        pre, act = gg.gmm_act(a, b1, group_sizes, fuse=True)
        none, only = gg.gmm_act(a, b1, group_sizes, fuse=True, keep_product=False)
        assert none is None and torch.equal(only, act)
        both = gg.gmm_gather(src, b1, group_sizes, act=gg.ACT_GELU_TANH, keep_product=False)
        assert (both is None) == (k % 64 != 0)
        assert both is None or (both[0] is None and torch.equal(both[1], act))
        for code in (0, 1):
            h = gg.gmm_glu(a, b1, b2, group_sizes, code, fuse=True)[2]
            none, none2, only = gg.gmm_glu(a, b1, b2, group_sizes, code, fuse=True, keep_product=False)
            assert none is None and none2 is None and torch.equal(only, h)
            got = gg.gmm_gather(src, b1, group_sizes, b2=b2, act=code, keep_product=False)
            assert got is None if k % 64 else torch.equal(got[2], h)
    # fp32: no such launch, the products come back
    pre, act = gg.gmm_act(x.float(), b1.float(), _sizes(groups, tokens, seed=1).cuda(), keep_product=False)
    assert pre.shape == act.shape


@pytest.mark.parametrize('groups,rows,k,n,skew', [(1, 1, 8, 8, False), (1, 1024, 128, 136, False), (3, 0, 64, 128, False),
                                                  (4, 257, 136, 120, False), (8, 8 * 63, 264, 1032, True), (64, 64 * 130, 256, 384, True),
                                                  (70, 70 * 40, 72, 264, True), (130, 900, 128, 2056, False),
                                                  (5, 5 * 256, 1032, 4616, False), (16, 16 * 257, 1024, 2056, True)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_gmm_tn_with_few_rows_per_expert(gg, groups, rows, k, n, skew, dtype):
    """Weight gradients with short reductions, on both sides of the line where the kernel for them takes over, alike and
    skewed experts, plain and on gathered rows, against fp32; rows of infinities past an expert's last (its neighbour's) must not
    reach it."""
    torch.manual_seed(rows + k)
    if skew:
        p = torch.arange(1, groups + 1).float() ** -1.2
        sizes = (p / p.sum() * rows).floor().long()
        sizes[0] += rows - int(sizes.sum())
        sizes = sizes[torch.randperm(groups)]
    else:
        sizes = _sizes(groups, rows, seed=k, empty=(0,) if groups > 2 and rows else ())
    a = torch.randn(rows, k, device='cuda').to(dtype)
    x = torch.randn(max(rows, 1), n, device='cuda').to(dtype)[:rows]
    b = x.clone()
    ends = torch.cumsum(sizes, 0)
    bad = int(torch.nonzero(sizes)[0]) if rows > 1 and int((sizes > 0).sum()) > 1 else -1
    if bad >= 0:
        b[int(ends[bad] - sizes[bad]):int(ends[bad])] = float('inf')
    keep = [e for e in range(groups) if e != bad]
    want = torch.stack([a[int(ends[e] - sizes[e]):int(ends[e])].float().t() @ b[int(ends[e] - sizes[e]):int(ends[e])].float()
                        for e in keep]) if keep else torch.zeros(0, k, n, device='cuda')
    got = gg.backend.gmm(a, b, sizes, trans_a=True)
    assert torch.isfinite(got[keep]).all() and (not keep or rel_err(got[keep], want) < TOL)
    assert not got[(sizes == 0).cuda()].any()
    if keep and float(want.abs().max()) > 0:
        assert max_block_err(got[keep], want) < TOL
    if rows and k > 128:   # one expert per token: row r is row order[r] of the tokens
        order = torch.randperm(rows, device='cuda').int()
        bins = ends.cuda().int()
        bin_ids = torch.repeat_interleave(torch.arange(groups), sizes).int().cuda()
        src = gg.GatheredRows(x, order, bin_ids, bins, None, 1, rows)
        assert torch.equal(gg.gmm_tn_gather(a, src, sizes.cuda()), gg.backend.gmm(a, x[order.long()], sizes, trans_a=True))


@pytest.mark.parametrize('groups,rows,k,n', [(70, 70 * 80, 504, 2568), (64, 64 * 300, 520, 1672), (9, 9 * 270, 4600, 2056), (12, 12 * 100, 768, 1032),
                                             (16, 16 * 300, 1160, 648), (40, 40 * 520, 2312, 584), (6, 6 * 1024, 1416, 520), (4, 4 * 280, 2056, 1032)])
@pytest.mark.parametrize('spread', ['alike', 'skewed'])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_gmm_tn_of_many_tiles(gg, groups, rows, k, n, spread, dtype):
    """Weight gradients of up to a few hundred rows per expert in launches of many tiles, block by block against fp32, and bit for bit
    those on gathered rows, which the general kernels form; an expert without rows."""
    torch.manual_seed(rows + k)
    if spread == 'alike':
        sizes = rows // groups + torch.randint(-20, 21, (groups,))
        sizes[1] += sizes[2]
        sizes[2] = 0
    else:
        sizes = _sizes(groups, rows, seed=k, empty=(0, groups - 2))
    rows = int(sizes.sum())
    a, b = torch.randn(rows, k, device='cuda').to(dtype), torch.randn(rows, n, device='cuda').to(dtype)
    got = gg.backend.gmm(a, b, sizes, trans_a=True)
    wide = gg.weight_gradient(a, b, sizes.cuda(), torch.float32)
    assert torch.equal(wide.to(dtype), got) and not got[(sizes == 0).cuda()].any()
    ends = torch.cumsum(sizes, 0)
    for e in range(groups):
        s = slice(int(ends[e] - sizes[e]), int(ends[e]))
        if sizes[e]:
            assert max_block_err(got[e], a[s].float().t() @ b[s].float()) < TOL
    bin_ids = torch.repeat_interleave(torch.arange(groups), sizes).int().cuda()
    src = gg.GatheredRows(b, torch.arange(rows, device='cuda').int(), bin_ids, ends.cuda().int(), None, 1, rows)
    assert torch.equal(gg.gmm_tn_gather(a, src, sizes.cuda()), got)


@pytest.mark.parametrize('groups,rows,k,n,kernel', [(70, 24, 520, 616, 3), (70, 24, 136, 1544, 1), (33, 100, 1032, 1032, 1), (33, 100, 1032, 1056, 3),
                                                    (80, 128, 1160, 1096, 1), (80, 129, 1160, 1096, 2), (80, 65, 1280, 1088, 2), (5, 513, 136, 2056, 3),
                                                    (54, 600, 176, 1544, 2)])
def test_gmm_tn_stores_of_whole_and_split_pieces(gg, groups, rows, k, n, kernel):
    """Weight gradients on both sides of the lines between the kernels for few rows per expert, each in the kernel the rule names, block by
    block against fp32 and bit for bit those on gathered rows; what lies around the product stays."""
    from megablocks_amd import _lib
    f = _lib.lib.mbx_debug_tn_kernel_by_rule
    f.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
    assert f(groups, groups * rows, k, n) == kernel
    torch.manual_seed(rows + n)
    sizes = torch.full((groups,), rows)
    sizes[0], sizes[1] = 2 * rows, 0
    a, b = torch.randn(groups * rows, k, device='cuda').bfloat16(), torch.randn(groups * rows, n, device='cuda').bfloat16()
    around = torch.full((groups * k * n + 2 * n,), 7.0, device='cuda', dtype=torch.bfloat16)
    got = around[n:-n].view(groups, k, n)
    gg.backend.gmm(a, b, sizes, trans_a=True, c=got)
    assert (around[:n] == 7).all() and (around[-n:] == 7).all() and not got[1].any()
    ends = torch.cumsum(sizes, 0)
    for e in range(groups):
        s = slice(int(ends[e] - sizes[e]), int(ends[e]))
        if sizes[e]:
            assert max_block_err(got[e], a[s].float().t() @ b[s].float()) < TOL
    bin_ids = torch.repeat_interleave(torch.arange(groups), sizes).int().cuda()
    src = gg.GatheredRows(b, torch.arange(groups * rows, device='cuda').int(), bin_ids, ends.cuda().int(), None, 1, groups * rows)
    assert torch.equal(gg.gmm_tn_gather(a, src, sizes.cuda()), got)


@pytest.mark.parametrize('groups,rows,k,n', [(1, 1, 8, 8), (3, 130, 64, 136), (5, 5 * 300, 264, 1032), (70, 900, 136, 256), (4, 4 * 1500, 392, 264),
                                             (8, 8 * 2100, 1024, 640), (2, 0, 64, 64)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_weight_gradients_of_fp32_weights(gg, groups, rows, k, n, dtype):
    """The fp32 weight gradient of 16-bit operands: rounded it is the 16-bit product bit for bit, and against fp64 it shows
    the error of an fp32 sum (2^-24 per term, random signs, a factor of four to spare).  Plain and on gathered rows."""
    torch.manual_seed(rows + n)
    sizes = _sizes(groups, rows, seed=k, empty=(0,) if groups > 2 and rows else ()).cuda()
    a = torch.randn(rows, k, device='cuda').to(dtype)
    x = torch.randn(rows, n, device='cuda').to(dtype)
    got = gg.weight_gradient(a, x, sizes, torch.float32)
    assert got.dtype == torch.float32 and torch.equal(got.to(dtype), gg.backend.gmm(a, x, sizes, trans_a=True))
    start = 0
    for e, c in enumerate(sizes.tolist()):
        want = a[start:start + c].double().t() @ x[start:start + c].double()
        assert rel_err(got[e].double(), want) <= 4 * 2.0 ** -24 * max(c, 16) ** 0.5 if c else not got[e].any()
        start += c
    assert gg.weight_gradient(a, x, sizes).dtype == dtype and gg.weight_gradient(a, x, sizes, dtype).dtype == dtype
    if rows and k > 128:
        order = torch.randperm(rows, device='cuda').int()
        bins = torch.cumsum(sizes, 0).int()
        bin_ids = torch.repeat_interleave(torch.arange(groups, device='cuda'), sizes.long()).int()
        src = gg.GatheredRows(x, order, bin_ids, bins, None, 1, rows)
        wide = src.weight_gradient(a, sizes, torch.float32)
        assert wide.dtype == torch.float32 and torch.equal(wide.to(dtype), gg.gmm_tn_gather(a, src, sizes))


@pytest.mark.parametrize('mlp', ['mlp', 'glu'])
@pytest.mark.parametrize('memopt', [False, True])
@pytest.mark.parametrize('top_k', [1, 4])
def test_autocast_gradients_of_fp32_experts(gg, mlp, memopt, top_k):
    """A layer with fp32 parameters under autocast: every gradient in fp32, the experts' without the rounding to bf16 the plain
    route gives them, and within one rounding of that route's."""
    from megablocks_amd.layers.arguments import Arguments
    from megablocks_amd.layers.dmoe import dMoE
    torch.manual_seed(3)
    kw = dict(activation_fn=torch.nn.functional.silu) if mlp == 'glu' else {}
    layer = dMoE(Arguments(hidden_size=136, ffn_hidden_size=264, moe_num_experts=8, moe_top_k=top_k, bias=False, mlp_type=mlp, mlp_impl='grouped',
                           memory_optimized_mlp=memopt, moe_loss_weight=0.0, fp16=False, bf16=False, device=torch.device('cuda'), **kw))
    x = torch.randn(200, 1, 136, device='cuda', requires_grad=True)
    grad = torch.randn(200, 1, 136, device='cuda').bfloat16()
    results = []
    for wide in (True, False):
        with pytest.MonkeyPatch.context() as patch:
            if not wide:
                patch.setattr(gg, '_wants_fp32', lambda *_: False)
            layer.zero_grad(set_to_none=True)
            x.grad = None
            with torch.autocast('cuda', dtype=torch.bfloat16):
                y = layer(x)
            y.backward(grad)
            results.append([x.grad] + [p.grad for p in layer.parameters()])
    assert torch.equal(results[0][0], results[1][0])
    rounded = 0
    for got, want in zip(*results):
        assert got.dtype == want.dtype == torch.float32
        assert torch.equal(got, want) or torch.equal(got.bfloat16().float(), want)
        rounded += not torch.equal(got, want)
    assert rounded == (3 if mlp == 'glu' else 2)


@pytest.mark.parametrize('groups,rows,k,n', [(64, 640, 64, 1032), (70, 70 * 40, 72, 1288), (300, 12000, 128, 8), (9, 9 * 39, 520, 7688),
                                             (8, 8 * 40 + 1, 192, 8456), (40, 40 * 30, 1032, 2056)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_gmm_nt_with_a_few_dozen_rows_per_expert(gg, groups, rows, k, n, dtype):
    """NT launches on both sides of the line where the kernel for them takes over, every form, against fp32; the forms' products
    equal bit for bit.  Experts of 0 to more than 64 rows; an infinite expert must not reach its neighbours."""
    torch.manual_seed(rows)
    sizes = _sizes(groups, rows, seed=rows, empty=(1,))
    ends = torch.cumsum(sizes, 0)
    a = torch.randn(rows, k, device='cuda').to(dtype)
    w, v = ((torch.randn(groups, n, k, device='cuda') / k ** 0.5).to(dtype) for _ in range(2))
    w[2] = float('inf')   # an expert's weights: its rows only
    keep = torch.ones(rows, 1, dtype=torch.bool, device='cuda')
    keep[int(ends[1]):int(ends[2])] = False
    zero = torch.zeros((), device='cuda')

    def check(got, want):
        got, want = (torch.where(keep, t.float(), zero) for t in (got, want))
        assert rel_err(got, want) < TOL and max_block_err(got, want, 8, 32) < 4 * TOL

    def same(x, y):
        return torch.equal(torch.where(keep, x.float(), zero), torch.where(keep, y.float(), zero))

    ref, ref_v = _ref_gpu(a, w, sizes, False, True), _ref_gpu(a, v, sizes, False, True)
    sizes = sizes.cuda()
    c = gg.backend.gmm(a, w, sizes, trans_b=True)
    check(c, ref)
    pre, act = gg.gmm_act(a, w, sizes, fuse=True)
    assert same(pre, c)
    check(act, torch.nn.functional.gelu(c.float(), approximate='tanh'))
    saved, saved2 = torch.randn(rows, n, device='cuda').to(dtype), torch.randn(rows, n, device='cuda').to(dtype)
    x = saved.float().requires_grad_(True)
    torch.nn.functional.gelu(x, approximate='tanh').backward(torch.where(keep, c.float(), zero))
    check(gg.gmm_dact(a, w, saved, sizes, fuse=True), x.grad)
    for code, fn in ((0, torch.nn.functional.silu), (1, lambda t: torch.nn.functional.gelu(t, approximate='tanh'))):
        x1, x2, h = gg.gmm_glu(a, w, v, sizes, code, fuse=True)
        assert same(x1, c)
        check(x2, ref_v)
        check(h, fn(x1.float()).to(dtype).float() * x2.float())
        p, q = saved.float().requires_grad_(True), saved2.float().requires_grad_(True)
        (fn(p) * q).backward(torch.where(keep, c.float(), zero))
        d1, d2 = gg.gmm_dglu(a, w, saved, saved2, sizes, code, fuse=True)
        check(d1, p.grad)
        check(d2, q.grad)
    if k % 64 == 0:
        order = torch.randperm(rows, device='cuda').int()
        bins = ends.cuda().int()
        bin_ids = torch.repeat_interleave(torch.arange(groups, device='cuda'), sizes.long()).int()
        tokens = torch.empty_like(a)
        tokens[order.long()] = a
        src = gg.GatheredRows(tokens, order, bin_ids, bins, None, 1, rows)
        assert same(gg.gmm_gather(src, w, sizes)[0], c)
        assert same(gg.gmm_gather(src, w, sizes, b2=v, act=1)[2], h)
        assert same(gg.gmm_gather(src, w, sizes, b2=v, act=1, keep_product=False)[2], h)


@pytest.mark.parametrize('tokens,experts,top_k,k,n,blocking', [
    (400, 64, 6, 128, 1288, 0), (640, 64, 2, 320, 1288, 0), (256, 128, 4, 64, 776, 0), (296, 40, 3, 192, 2056, 0), (75, 12, 5, 64, 5896, 0),
    # padded rows: expert e's start at a multiple of 128 in the product and not in the list of assignments
    (12, 80, 2, 128, 1800, 128), (6, 64, 3, 64, 1544, 128),
])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_gathered_products_of_a_few_dozen_rows_per_expert(gg, tokens, experts, top_k, k, n, blocking, dtype):
    """The kernel for a few dozen rows per expert (up to 40 on average, more 64 x 256 tiles than compute units) reading
    its rows through the assignments: several experts per token, padded and not, every form, against the gathered copy and
    the product on it, bit for bit."""
    indices, bin_ids, bins, padded, tpe = _routing(tokens, experts, top_k, seed=tokens, blocking=blocking)
    sizes = torch.diff(padded, prepend=padded.new_zeros(1)) if blocking else tpe
    rows = int(sizes.sum())
    assert rows <= 40 * experts and experts * ((n + 255) // 256) * 0.95 > 256
    x = torch.randn(tokens, k, device='cuda').to(dtype)
    w1, v1 = ((torch.randn(experts, n, k, device='cuda') / k ** 0.5).to(dtype) for _ in range(2))
    src = gg.GatheredRows(x, indices, bin_ids, bins, padded, top_k, rows)
    a = src.materialize()
    (c,) = gg.gmm_gather(src, w1, sizes)
    assert torch.equal(c, gg.backend.gmm(a, w1, sizes, trans_b=True))
    assert max_block_err(c, _ref_gpu(a, w1, sizes.cpu(), False, True), 8, 32) < 4 * TOL
    pre, act = gg.gmm_gather(src, w1, sizes, act=gg.ACT_GELU_TANH)
    want_pre, want_act = gg.gmm_act(a, w1, sizes, fuse=True)
    assert torch.equal(pre, c) and torch.equal(want_pre, c) and torch.equal(act, want_act)
    assert torch.equal(gg.gmm_gather(src, w1, sizes, act=gg.ACT_GELU_TANH, keep_product=False)[1], act)
    for code in (0, 1):
        got, want = gg.gmm_gather(src, w1, sizes, b2=v1, act=code), gg.gmm_glu(a, w1, v1, sizes, code, fuse=True)
        assert all(torch.equal(p, q) for p, q in zip(got, want)) and torch.equal(got[0], c)
        assert torch.equal(gg.gmm_gather(src, w1, sizes, b2=v1, act=code, keep_product=False)[2], got[2])


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_gelu_forward_is_the_epilogues(gg, dtype):
    """The pass of its own gives what the first product's epilogue stores, for every finite 16-bit value; from an address or of a
    size it does not take, torch's values."""
    x = torch.arange(-32768, 32768, dtype=torch.int32, device='cuda').to(torch.int16).view(dtype)
    x = torch.where(torch.isfinite(x), x, torch.zeros_like(x)).view(-1, 8)
    pre, act = gg.gmm_act(x, torch.eye(8, device='cuda').to(dtype)[None], torch.tensor([x.shape[0]]), fuse=True)
    assert torch.equal(pre, x) and torch.equal(gg.gelu_forward(pre), act)
    for odd in (pre.flatten()[1:9], pre.flatten()[:7], pre[:, ::2], pre.float()):
        assert torch.equal(gg.gelu_forward(odd), torch.nn.functional.gelu(odd, approximate='tanh'))
    assert gg.gelu_forward(pre[:0]).shape == (0, 8)
