"""The direct path of the Muon step (csrc/muon_direct.hip): on the GPU bit for
bit against mamw_muon_step on each matrix alone, at the edges of its tiles,
fragments and prep units; on the CPU its argument checks, the choice between
the two paths and the merging of launch groups.

No tolerance: every output element sums the same products in the same order
under either path (one chain of 32x32x16 MFMAs, k ascending), and the epilogues
round at the same places."""

import ctypes
import types

import pytest
import torch

from triton_muon_adamw import _lib
from triton_muon_adamw.muon import hip_muon
from triton_muon_adamw.muon.hip_muon import scaled_lr

COEFFS = (3.4445, -4.7750, 2.0315)
F32, BF16 = torch.float32, torch.bfloat16


def _arr(mats):
    arr = (_lib.MuonMatrix * len(mats))()
    for i, (p, g, m, u) in enumerate(mats):
        flags = (_lib.BF16_PARAM if p.dtype == BF16 else 0) | (_lib.BF16_GRAD if g.dtype == BF16 else 0)
        arr[i] = _lib.MuonMatrix(p.data_ptr(), g.data_ptr(), m.data_ptr(), u.data_ptr() if u is not None else None,
                                 *p.shape, scaled_lr(2e-2, "original", *p.shape), flags)
    return arr


def _make(shapes, dev, pd, gd, shift, with_update):
    """[param, grad, momentum, update] per shape; `shift`: each starts one element past an aligned address."""
    gen = torch.Generator(device=dev).manual_seed(21)
    out = []
    for r, c in shapes:
        def t(std, dtype):
            flat = torch.empty(r * c + shift, device=dev).normal_(0.0, std, generator=gen).to(dtype)
            return flat[shift:].view(r, c)
        out.append([t(0.02, pd), t(1e-3, gd), t(1e-3, F32), torch.zeros((r, c), device=dev) if with_update else None])
    return out


# one fragment and less; 32- and 64-wide edges; several prep units, ragged; all
# in one launch, tall and wide mixed; one shape (addresses from the block
# number); enough 64-wide tiles for the wide tile on the updates (18 x 24 = 432)
# and on every product (32 x 33 / 2 = 528)
SETS = [
    [(1, 5), (5, 1), (1, 1), (31, 33), (32, 64), (33, 65), (64, 63), (65, 128), (129, 127)],
    [(10, 517), (517, 1003), (1003, 785)],
    [(256, 512)] * 3,
    [(512, 256), (256, 512)],
    [(1100, 1500)],
    [(2048, 2000)],
    [(192, 448)] * 33 + [(448, 192)] * 31,  # a full table
]


@pytest.mark.gpu
@pytest.mark.parametrize("shapes", SETS, ids=lambda s: f"{len(s)}x{s[0][0]}x{s[0][1]}")
@pytest.mark.parametrize("pd,gd,shift,ns_steps,nesterov", [(F32, F32, 0, 5, 1), (BF16, BF16, 0, 2, 1),
                                                           (F32, BF16, 1, 1, 0), (BF16, F32, 1, 3, 1)])
def test_direct_equals_staged(gpu, shapes, pd, gd, shift, ns_steps, nesterov):
    lib = _lib.load()
    stream = torch.cuda.current_stream(gpu).cuda_stream
    hyper = (2e-2, 0.1, 0.95, nesterov, *COEFFS, ns_steps, 1e-7)
    mine, ref = (_make(shapes, gpu, pd, gd, shift, ns_steps != 2) for _ in range(2))
    arr = _arr(mine)
    nbytes = hip_muon._direct_workspace_bytes(arr, len(shapes), ns_steps)
    ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=gpu)  # NaN wherever it is read unwritten
    _lib.check(lib.mamw_muon_direct_step(arr, len(shapes), *hyper, ws.data_ptr(), nbytes, None, None, stream), "direct")
    for x in ref:
        n = hip_muon._workspace_bytes(1, *x[0].shape, ns_steps)
        w1 = torch.empty(n, dtype=torch.uint8, device=gpu)
        _lib.check(lib.mamw_muon_step(_arr([x]), 1, *hyper, w1.data_ptr(), n, stream), "staged")
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(zip(mine, ref)):
        for k, what in ((0, "param"), (2, "momentum"), (3, "update")):
            if a[k] is not None:
                assert torch.equal(a[k], b[k]), (i, shapes[i], what)


# A last round of few 256-wide tiles as 128-wide ones (muon.hip launch_gemm):
# every product of one 2048 x 2300 (36 and 72 tiles, no full round); 260
# symmetric tiles, four after a full round, lower-triangle A and B; 360 (104
# after a full round) with ragged edges and both orientations.
@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [[(2048, 2300)], [(1024, 1280)] * 26, [(2100, 2100)] * 4 + [(2100, 2100)] * 4],
                         ids=lambda s: f"{len(s)}x{s[0][0]}x{s[0][1]}")
def test_split_last_round_equals_direct(gpu, shapes):
    """Bit for bit against the direct path, which has neither tiles nor lower triangles in common with it."""
    lib = _lib.load()
    stream = torch.cuda.current_stream(gpu).cuda_stream
    hyper = (2e-2, 0.1, 0.95, 1, *COEFFS, 3, 1e-7)
    mine, ref = (_make(shapes, gpu, F32, F32, 0, True) for _ in range(2))
    n = hip_muon._workspace_bytes(len(shapes), *shapes[0], 3)
    ws = torch.full((n,), 0xFF, dtype=torch.uint8, device=gpu)
    _lib.prof_start()
    _lib.check(lib.mamw_muon_step(_arr(mine), len(shapes), *hyper, ws.data_ptr(), n, stream), "staged")
    _lib.prof_stop()
    recs = [r for r in _lib.prof_collect() if r["kernel"].startswith("ns_gemm")]
    assert len(recs) == 9  # one per product, named after its whole rounds where it has any
    assert {r["variant"] // 8 for r in recs if r["kernel"] in ("ns_gemm_kernel:gram", "ns_gemm_kernel:poly")} == {
        128 if len(shapes) == 1 else 256}
    arr = _arr(ref)
    n = hip_muon._direct_workspace_bytes(arr, len(shapes), 3)
    ws = torch.empty(n, dtype=torch.uint8, device=gpu)
    _lib.check(lib.mamw_muon_direct_step(arr, len(shapes), *hyper, ws.data_ptr(), n, None, None, stream), "direct")
    torch.cuda.synchronize()
    for a, b in zip(mine, ref):
        for k in (0, 2, 3):
            assert torch.equal(a[k], b[k])


@pytest.mark.gpu
@pytest.mark.parametrize("inf", [0.0, 1.0])
def test_direct_gradient_scaler_step(gpu, inf):
    """grad_scale divides the gradients; a non-zero found_inf leaves everything as it was."""
    lib = _lib.load()
    stream = torch.cuda.current_stream(gpu).cuda_stream
    hyper = (2e-2, 0.1, 0.95, 1, *COEFFS, 5, 1e-7)
    shapes = [(100, 300), (300, 100), (64, 64)]
    mine, ref, start = (_make(shapes, gpu, F32, F32, 0, True) for _ in range(3))
    scale, found = torch.full((), 3.0, device=gpu), torch.full((), inf, device=gpu)
    arr = _arr(mine)
    nbytes = hip_muon._direct_workspace_bytes(arr, 3, 5)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=gpu)
    _lib.check(lib.mamw_muon_direct_step(arr, 3, *hyper, ws.data_ptr(), nbytes, scale.data_ptr(), found.data_ptr(),
                                         stream), "direct")
    for x in ref:
        n = hip_muon._workspace_bytes(1, *x[0].shape, 5)
        w1 = torch.empty(n, dtype=torch.uint8, device=gpu)
        _lib.check(lib.mamw_muon_step_amp(_arr([x]), 1, *hyper, w1.data_ptr(), n, scale.data_ptr(), found.data_ptr(),
                                          stream), "staged")
    torch.cuda.synchronize()
    for a, b, s in zip(mine, ref, start):
        for k in (0, 2, 3):
            assert torch.equal(a[k], b[k])
            assert torch.equal(a[k], s[k]) == (inf != 0.0)


def _mats(specs):
    arr = (_lib.MuonMatrix * len(specs))()
    for i, (r, c) in enumerate(specs):
        base = (i + 1) << 36
        arr[i] = _lib.MuonMatrix(base, base + (1 << 34), base + (2 << 34), None, r, c, 1e-3, 0)
    return arr


def _bytes(arr, n, steps=5):
    b = ctypes.c_size_t()
    return _lib.load().mamw_muon_direct_workspace_bytes(arr, n, steps, ctypes.byref(b)), b.value


def _step(arr, n, ws=1 << 45, ws_bytes=1 << 40, steps=5):
    return _lib.load().mamw_muon_direct_step(arr, n, 1e-3, 0.1, 0.95, 1, *COEFFS, steps, 1e-7, ws, ws_bytes, None,
                                             None, None)


def test_direct_rejects_before_hip():
    NULL, COUNT, SHAPE, ALIGN, WS, HYPER, ALIAS = -1, -2, -4, -5, -6, -7, -9
    ok = [(10, 517), (517, 1003)]
    st, need = _bytes(_mats(ok), 2)
    # the table, then X^T twice and X, A and B, the unit sums, per matrix
    rup = lambda x, t: -(-x // t) * t  # noqa: E731
    expect = 64 * 64
    for r, c in ok:
        mp, np_ = rup(min(r, c), 64), rup(max(r, c), 64)
        expect += rup(6 * mp * np_ + 4 * mp * mp + 4 * (rup(r, 128) // 32) * (rup(c, 128) // 128), 256)
    assert (st, need) == (0, expect)
    assert _bytes(_mats(ok), 0)[0] == COUNT and _bytes(_mats([(4, 4)] * 65), 65)[0] == COUNT
    assert _bytes(_mats(ok), 2, steps=0)[0] == HYPER and _bytes(_mats(ok), 2, steps=100)[0] == HYPER
    assert _bytes(_mats([(0, 4)]), 1)[0] == SHAPE and _bytes(_mats([(8192, 8256)]), 1)[0] == SHAPE
    # padded to 128: 2^26 elements, and twice as many (too many prep units for one block to sum)
    assert _bytes(_mats([(1, 1 << 19)]), 1)[0] == 0 and _bytes(_mats([(1, 1 << 20)]), 1)[0] == SHAPE
    assert _step(_mats(ok), 2, ws_bytes=need - 1) == WS and _step(_mats(ok), 2, ws=None) == WS
    assert _step(_mats(ok), 2, ws=(1 << 45) + 64) == WS
    for field, value, code in (("param", None, NULL), ("flags", 4, HYPER), ("momentum", (1 << 45) + 256, ALIAS),
                               ("grad", (2 << 36) + 2, ALIGN), ("param", 1 << 36, ALIAS)):
        arr = _mats(ok)
        setattr(arr[1], field, value)
        assert _step(arr, 2) == code, field


def test_direct_choice():
    """Small groups go direct, groups that fill the GPU with staged tiles do not; a set of classes goes as one."""
    pays = hip_muon.direct_pays
    for shape, count in (((512, 2048), 2), ((3072, 768), 1), ((10, 517), 32), ((1536, 1536), 1), ((1024, 4096), 1)):
        assert pays(*shape, count, 256, 5), (shape, count)
    for shape, count in (((512, 2048), 16), ((768, 3072), 12), ((1024, 2048), 8), ((4096, 4096), 1),
                         ((14336, 4096), 1), ((8192, 8256), 1)):
        assert not pays(*shape, count, 256, 5), (shape, count)
    assert not pays(64, 64, 1, 256, 0)  # ns_steps = 0 has no product to run
    both = hip_muon.direct_set_pays
    assert both(((785, 1003, 1), (517, 1003, 1), (10, 517, 1)), 256, 5)
    assert both(((256, 1024, 4), (256, 768, 2), (256, 256, 2)), 256, 5)
    assert not both(((768, 3072, 24), (768, 2304, 12), (768, 768, 12)), 256, 5)
    assert not both(((1024, 2048, 1), (2048, 4096, 1), (4096, 4096, 1), (1024, 4096, 1)), 256, 5)


def test_ns_direct_choice():
    """Standalone products against the row-major staged kernels, which never
    split a last round of few 256-wide tiles (GPU times of both paths in
    ``ns_direct_pays``): one round of 36 to 55 symmetric tiles, of 64 update
    tiles, and rows that padding takes to 2048."""
    GRAM, POLY, UPDATE, STEP = range(4)
    pays = hip_muon.ns_direct_pays
    for op, m, n in ((GRAM, 1024, 4096), (GRAM, 2048, 8192), (GRAM, 2177, 4096), (GRAM, 2304, 4096),
                     (GRAM, 2560, 4096), (GRAM, 2560, 8192), (GRAM, 2000, 8192), (POLY, 1024, 1024),
                     (POLY, 2304, 2304), (POLY, 2560, 2560), (POLY, 3072, 3072), (UPDATE, 768, 3001),
                     (UPDATE, 2048, 2048), (STEP, 512, 512), (STEP, 2048, 4000), (STEP, 2304, 4096),
                     (STEP, 2560, 2560)):
        assert pays(op, m, n, 256), (op, m, n)
    for op, m, n in ((GRAM, 4096, 4096), (POLY, 4096, 4096), (UPDATE, 2048, 8192), (STEP, 4096, 4096),
                     (GRAM, 8256, 8256)):
        assert not pays(op, m, n, 256), (op, m, n)


def test_merged_launches():
    """Groups go out together up to the table's size and only where no matrix
    writes what another reads or writes."""
    def call(specs, group, first):
        arr = (_lib.MuonMatrix * len(specs))()
        for i, (r, c) in enumerate(specs):
            base = (first + i + 1) << 36
            arr[i] = _lib.MuonMatrix(base, base + (1 << 34), base + (2 << 34), None, r, c, 1e-3, 0)
        return hip_muon._Call("d0", arr, len(specs), 0, 8, 16, group, True)

    runs = lambda calls: [[c.group for c in r] for r in hip_muon._merge(calls)]  # noqa: E731
    a, b, c = call([(8, 16)] * 30, 0, 0), call([(16, 32)] * 30, 1, 30), call([(4, 4)] * 5, 2, 60)
    assert runs([a, b, c]) == [[0, 1], [2]]
    a, b = call([(8, 16)], 0, 0), call([(16, 32)], 1, 1)
    assert runs([a, b]) == [[0, 1]]
    b.arr[0].grad = a.arr[0].grad  # two readers
    assert runs([a, b]) == [[0, 1]]
    b.arr[0].grad = a.arr[0].param  # one matrix's gradient is the other's parameter
    assert runs([a, b]) == [[0], [1]]
    b = call([(16, 32)], 1, 1)
    b.arr[0].param = a.arr[0].param + 8 * 16 * 4 - 4  # the last element shared
    assert runs([a, b]) == [[0], [1]]
    b.arr[0].param += 4
    assert runs([a, b]) == [[0, 1]]


@pytest.fixture
def planner(monkeypatch):
    """plan(shapes, limit=None, **attributes) -> the HipMuon with its launches
    planned, on the CPU: 256 CUs, the library's own sizes and choices."""
    props = types.SimpleNamespace(multi_processor_count=256, total_memory=288 << 30)
    streams = []
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda dev: props)
    monkeypatch.setattr(_lib, "require_gpu_tensor", lambda t, name: None)
    monkeypatch.setattr(_lib, "raw_stream", lambda dev: 0)
    monkeypatch.setattr(_lib, "side_streams", lambda dev, n: streams.append(n) or [f"side{i}" for i in range(n)])

    def plan(shapes, limit=None, **attributes):
        params = [torch.nn.Parameter(torch.zeros(s)) for s in shapes]
        for p in params:
            p.grad = torch.zeros_like(p)
        opt = hip_muon.HipMuon(params)
        opt.workspace_limit_bytes = limit
        for k, v in attributes.items():
            setattr(opt, k, v)
        opt._build_calls(params)
        return opt

    plan.streams = streams
    return plan


@pytest.mark.parametrize("limit_mib", [None, 60, 20, 6, 1])
@pytest.mark.parametrize("in_order", [False, True])
def test_launches_keep_to_the_workspace_limit(planner, limit_mib, in_order):
    """Merged or not, direct or staged: no launch's workspace is over the limit
    unless one matrix alone needs it on the staged path, and every matrix goes
    out once, with room for it."""
    shapes = [(256, 1024)] * 32 + [(256, 768)] * 2 + [(128, 8192), (8192, 128)]
    limit = None if limit_mib is None else limit_mib << 20
    opt = planner(shapes, limit, **({"concurrent_flops_limit": 0.0} if in_order else {}))
    assert sum(x.n for x in opt._launches) == len(shapes)
    assert len({e.param for x in opt._launches for e in x.arr}) == len(shapes)
    for x in opt._launches:
        one = {hip_muon._workspace_bytes(1, e.rows, e.cols, 5) for e in x.arr}
        need = (hip_muon._direct_workspace_bytes(x.arr, x.n, 5) if x.direct
                else hip_muon._workspace_bytes(x.n, x.arr[0].rows, x.arr[0].cols, 5))
        assert opt._ws[x.ws_key].numel() >= need
        if limit is not None:
            assert need <= limit or not x.direct and x.n == 1 and one == {need}
    if not in_order and limit is None:  # 36 matrices, one launch
        assert [(x.n, x.direct, x.lane) for x in opt._launches] == [(36, True, None)]


def test_streams_for_staged_classes_only(planner):
    """Classes that go out together on the caller's stream make no side streams
    (a thread keeps those it makes); staged classes run on the ones made."""
    opt = planner([(256, 1024)] * 4 + [(256, 768)] * 2 + [(256, 256)] * 2)
    assert opt._concurrent and [(x.n, x.direct, x.lane) for x in opt._launches] == [(8, True, None)]
    assert planner.streams == [] and opt._lanes == {}
    opt = planner([(1024, 2048), (2048, 4096), (4096, 4096), (4096, 1024)])
    assert opt._concurrent and not any(x.direct for x in opt._launches)
    lanes = [x.lane for x in opt._launches]
    assert planner.streams == [2] and lanes[0] is None and set(lanes[1:]) == {"side0", "side1"}
    assert len({x.ws_key for x in opt._launches}) == 4


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["current", "side", "graph"])
def test_merged_classes_equal_staged_in_order(gpu, monkeypatch, how):
    """Shape classes that go out as one direct launch, on the caller's stream:
    the bits of staged classes one after another, also under a side stream and
    in a graph that is replayed between eager work."""
    shapes = [(256, 512)] * 3 + [(512, 256)] * 2 + [(384, 384)] * 2 + [(128, 640), (10, 517)]
    start = _make(shapes, gpu, F32, F32, 0, False)
    grads = [_make(shapes, gpu, F32, F32, 0, False)[i][1] * (1 + i / 7) for i in range(len(shapes))]

    def optimizer():
        params = [torch.nn.Parameter(p.clone()) for p, _, _, _ in start]
        opt = hip_muon.HipMuon(params, lr=2e-2, coeffs=COEFFS)
        for p, g, (_, _, m, _) in zip(params, grads, start):
            p.grad = g.clone()
            opt.momentum[p].copy_(m)
        return params, opt

    params, opt = optimizer()
    rparams, ropt = optimizer()
    ropt.concurrent_flops_limit = 0.0

    def reference_step():
        with monkeypatch.context() as m:
            m.setattr(hip_muon, "direct_pays", lambda *_: False)
            ropt.step()
        assert not any(x.direct for x in ropt._launches)

    def compare():
        torch.cuda.synchronize()
        for p, q in zip(params, rparams):
            assert torch.equal(p, q) and torch.equal(opt.momentum[p], ropt.momentum[q])

    opt.step()
    assert opt._concurrent and [(x.n, x.direct, x.lane) for x in opt._launches] == [(9, True, None)]
    reference_step()
    compare()
    if how == "graph":
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            opt.step()
    side = torch.cuda.Stream(device=gpu) if how == "side" else torch.cuda.current_stream(gpu)
    for i in range(4):
        for p, q in zip(params, rparams):  # other gradients in the same buffers
            p.grad.mul_(-1.25)
            q.grad.mul_(-1.25)
        side.wait_stream(torch.cuda.current_stream(gpu))
        with torch.cuda.stream(side):
            graph.replay() if how == "graph" else opt.step()
        torch.cuda.current_stream(gpu).wait_stream(side)
        reference_step()
        compare()


# ---- Standalone products ----------------------------------------------------

def _ns_inputs(m, n, dev):
    gen = torch.Generator(device=dev).manual_seed(31)
    x = (torch.empty((m, n), device=dev).normal_(generator=gen) / (m**0.5 + n**0.5)).bfloat16()
    s = torch.empty((m, m), device=dev).normal_(generator=gen) / m
    return x, (s + s.T).bfloat16()


def _ns_call(op, x, s, out):
    a, b, c = COEFFS
    {0: lambda: hip_muon.solve_ns_kernel_1(x, out), 1: lambda: hip_muon.solve_ns_kernel_2(s, b, c, out),
     2: lambda: hip_muon.solve_ns_kernel_3(x, s, a, out), 3: lambda: hip_muon.newton_shultz_step(x, a, b, c, out)}[op]()


# single elements; fragment and tile edges; rows of 16-byte chunks or not; more
# rows than columns; the 64-wide tile on the symmetric products (2048) and on
# the update only (1280 x 1300)
NS_SHAPES = [(1, 1), (5, 3), (31, 40), (64, 64), (65, 33), (10, 517), (517, 10), (333, 777), (128, 384), (1280, 1300),
             (2048, 136)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", NS_SHAPES, ids=str)
def test_ns_direct_equals_staged(gpu, shape, monkeypatch):
    """Bit for bit (same sums, same order), also with out over the input, which is packed first."""
    x, s = _ns_inputs(*shape, gpu)
    for op in range(4):
        out = [torch.full((shape[0], shape[0]) if op < 2 else shape, 7.0, dtype=BF16, device=gpu) for _ in range(2)]
        for o, direct in zip(out, (True, False)):
            monkeypatch.setattr(hip_muon, "ns_direct_pays", lambda *_, d=direct: d)
            _ns_call(op, x, s, o)
        assert torch.equal(*out), op
        src = s if op == 1 else x
        if out[0].shape == src.shape:
            own = src.clone()
            monkeypatch.setattr(hip_muon, "ns_direct_pays", lambda *_: True)
            _ns_call(op, own if op != 1 else x, own if op == 1 else s, own)
            assert torch.equal(own, out[1]), op


@pytest.mark.gpu
def test_ns_outputs_of_any_kind(gpu):
    """What the copy into ``out`` took, it takes: other types and strides; what it refused is refused."""
    x, s = _ns_inputs(96, 200, gpu)
    for op in range(4):
        shape = (96, 96) if op < 2 else (96, 200)
        ref = torch.empty(shape, dtype=BF16, device=gpu)
        version = ref._version
        _ns_call(op, x, s, ref)
        assert ref._version > version  # an in-place write, as autograd counts them
        wide = torch.zeros((shape[0], shape[1] + 3), dtype=BF16, device=gpu)
        f32 = torch.empty(shape, device=gpu)
        for o in (wide[:, 1:-2], f32, torch.empty(shape[::-1], dtype=BF16, device=gpu).T):
            _ns_call(op, x, s, o)
            assert torch.equal(o.to(BF16), ref), op
        assert not wide[:, 0].any() and not wide[:, -2:].any()
        _ns_call(op, x.T.contiguous().T, s.T.contiguous().T, f32)  # strided inputs
        assert torch.equal(f32.to(BF16), ref)
        leaf = torch.zeros(shape, dtype=BF16, device=gpu, requires_grad=True)
        with pytest.raises(RuntimeError):
            _ns_call(op, x, s, leaf)
        with pytest.raises(RuntimeError):
            _ns_call(op, x, s, torch.empty((shape[0], shape[1] + 1), dtype=BF16, device=gpu))
    flat = torch.zeros(128 * 128 + 1, dtype=BF16, device=gpu)
    with pytest.raises(ValueError):  # unpadded and misaligned
        hip_muon.solve_ns_kernel_1(flat[1:].view(128, 128), torch.empty((128, 128), dtype=BF16, device=gpu))


def test_ns_direct_leaves_other_tensors_to_the_copy(monkeypatch):
    """Outputs and inputs of a subclass (their own copy_ runs) and calls in
    forward mode (copy_ clears the output's tangent) do not go past it."""
    class Sub(torch.Tensor):
        pass

    monkeypatch.setattr(torch.cuda, "get_device_properties",
                        lambda dev: types.SimpleNamespace(multi_processor_count=256))
    reached = []
    monkeypatch.setattr(hip_muon, "ns_direct_pays", lambda *_: reached.append(1))  # None: not direct
    x, s, out = torch.zeros(96, 200, dtype=BF16), torch.zeros(96, 96, dtype=BF16), torch.zeros(96, 200, dtype=BF16)

    def call(x=x, s=s, out=out):
        del reached[:]
        assert not hip_muon._ns_direct(2, x, s, out, 1.0, 0.0, 0.0)
        return bool(reached)

    assert call() and call(x=torch.nn.Parameter(x)) and call(out=torch.nn.Parameter(out, requires_grad=False))
    assert not call(out=out.as_subclass(Sub)) and not call(x=x.as_subclass(Sub)) and not call(s=s.as_subclass(Sub))
    with torch.autograd.forward_ad.dual_level():
        assert not call(out=torch.autograd.forward_ad.make_dual(out, torch.ones_like(out)))
    assert call()


@pytest.mark.gpu
def test_ns_output_with_a_tangent(gpu):
    """Forward mode: writing the output clears its tangent, as any in-place copy of a constant does."""
    x, s = _ns_inputs(96, 200, gpu)
    for op in range(4):
        shape = (96, 96) if op < 2 else (96, 200)
        ref = torch.empty(shape, dtype=BF16, device=gpu)
        _ns_call(op, x, s, ref)
        with torch.autograd.forward_ad.dual_level():
            out = torch.autograd.forward_ad.make_dual(torch.zeros_like(ref), torch.ones_like(ref))
            _ns_call(op, x, s, out)
            primal, tangent = torch.autograd.forward_ad.unpack_dual(out)
            assert torch.equal(primal, ref) and (tangent is None or not tangent.any()), op


def test_ns_direct_rejects_before_hip():
    NULL, SHAPE, ALIGN, WS, HYPER, ALIAS = -1, -4, -5, -6, -7, -9
    lib = _lib.load()
    n = ctypes.c_size_t()
    assert lib.mamw_ns_direct_workspace_bytes(100, 300, ctypes.byref(n)) == 0
    need = n.value
    X, S, O, W = 1 << 36, 2 << 36, 3 << 36, 4 << 36

    def call(op=3, x=X, s=S, o=O, m=100, k=300, ws=W, nb=need):
        return lib.mamw_ns_direct(op, x, s, o, m, k, *COEFFS, ws, nb, None)

    assert call(op=4) == HYPER and call(op=-1) == HYPER
    assert call(m=0) == SHAPE and call(k=1 << 21) == SHAPE and call(m=8256, k=8) == SHAPE
    assert call(x=None) == NULL and call(o=None) == NULL and call(op=2, s=None) == NULL
    assert call(x=X + 1) == ALIGN and call(o=O + 1) == ALIGN and call(op=2, s=S + 1) == ALIGN
    assert call(ws=None) == WS and call(ws=W + 64) == WS and call(nb=need - 1) == WS
    assert call(x=W + 256) == ALIAS and call(o=W + 256) == ALIAS and call(op=2, s=W + 256) == ALIAS
