"""spc_sparse_conv_products (a 27-tap conv as one dense product per source
row and tap, then a sum over every output row's table entries) against the
same sums in F64, at the edges of its tiles: source rows around 256, column
blocks that fill, straddle and leave part of the 256-column tiles, one
64-channel stage and several, one output row, tables with missing taps and
out-of-range entries, and each epilogue.

Bound per element: the F32 sums (27 cin products, any order) are within
gamma = 27 cin 2^-24 of the F64 one relative to the sum of magnitudes, and
the result is rounded once to the feature dtype (u = 2^-8 / 2^-11)."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def _setup(n_in, n_out, cin, cout, dt, seed):
    import torch

    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s, std=1.0: (torch.randn(s, generator=g, device="cuda") * std).to(dt)  # noqa: E731
    x, w, b = r(n_in, cin), r(cout, 27, cin, std=(27 * cin) ** -0.5), r(cout, std=0.1)
    # a third missing: sentinels past the end and negative entries
    idx = torch.randint(-n_in // 4 - 1, n_in + n_in // 4 + 1, (n_out, 27), generator=g,
                        device="cuda", dtype=torch.int32)
    return x, w, b, idx


def _ref(x, w, b, idx):
    """F64 sums and the sums of magnitudes."""
    import torch

    n_in = x.shape[0]
    ok = (idx >= 0) & (idx < n_in)
    y = b.double().expand(idx.shape[0], -1).clone()
    mag = y.abs()
    for o in range(27):
        src = torch.where(ok[:, o, None], x[idx[:, o].clamp(0, n_in - 1).long()].double(), 0.0)
        y += src @ w[:, o].double().t()
        mag += src.abs() @ w[:, o].double().abs().t()
    return y, mag


@pytest.mark.parametrize("n_in,n_out,cin,cout", [
    (1, 1, 64, 32), (255, 700, 64, 128), (256, 1000, 128, 64), (257, 1000, 192, 96),
    (700, 64, 256, 160), (1500, 4001, 320, 128), (40, 3000, 64, 256)])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_products_conv(spc, dev, dtype, n_in, n_out, cin, cout):
    import torch

    print(f"[case] products conv {dtype} {n_in}->{n_out} rows {cin}->{cout}", flush=True)
    nat = spc._native
    dt, u = {"bf16": (torch.bfloat16, 2.0 ** -8), "f16": (torch.float16, 2.0 ** -11)}[dtype]
    x, w, b, idx = _setup(n_in, n_out, cin, cout, dt, n_in + cin)
    pw = nat.pack_weights(w)
    y = nat.sparse_conv_products(x, pw, b, idx.reshape(-1), n_out=n_out)
    ref, mag = _ref(x, w, b, idx)
    # (2^-25: half the smallest f16 subnormal)
    bound = mag * (27 * cin * 2.0 ** -24) + (ref.abs() + mag * (27 * cin * 2.0 ** -24)) * u + 2.0 ** -25
    assert bool(((y.double() - ref).abs() <= bound).all())
    # the epilogues act on the rounded rows as the conv's do
    g = torch.Generator(device="cuda").manual_seed(3)
    rows = torch.randint(-2, 34, (n_out,), generator=g, device="cuda", dtype=torch.int32)
    res = torch.randn((32, cout), generator=g, device="cuda").to(dt)
    yr = nat.sparse_conv_products(x, pw, b, idx.reshape(-1), n_out=n_out, residual=res,
                                  residual_rows=rows)
    ok = (rows >= 0) & (rows < 32)
    add = torch.where(ok[:, None], res[rows.clamp(0, 31).long()], torch.zeros_like(res[:1]))
    assert torch.equal(yr, y + add)
    full = torch.randn((n_out, cout), generator=g, device="cuda").to(dt)
    assert torch.equal(nat.sparse_conv_products(x, pw, b, idx.reshape(-1), n_out=n_out,
                                                residual=full), y + full)
    if cout in (32, 64, 128):
        coords = torch.zeros((n_out, 4), dtype=torch.int32, device=dev)
        coords[n_out // 2:, 0] = 1
        sc, sh = (torch.randn((2, cout), generator=g, device="cuda").to(dt) for _ in range(2))
        yn = nat.sparse_conv_products(x, pw, b, idx.reshape(-1), n_out=n_out,
                                      norm_mod=(sc, sh, coords, 1e-6))
        ref = nat.layernorm_mod_silu(y, sc, sh, coords, eps=1e-6)
        # the same steps; where the two kernels' F32 statistics differ in the
        # last place a rounding to dt may flip: half a spacing each of the
        # norm, the product and the sum, then of silu (slope <= 1.1)
        k = coords[:, 0].long()
        nrm = torch.nn.functional.layer_norm(y.double(), (cout,), eps=1e-6).abs()
        m = nrm * (1 + sc[k].double().abs()) + sh[k].double().abs()
        assert bool(((yn.double() - ref.double()).abs() <= 2 * 4 * u * m + 2.0 ** -24).all())
        assert float((yn != ref).float().mean()) <= 0.01


@pytest.mark.parametrize("at", [0, 1, 2, 3])
def test_products_conv_bias_at_any_element(spc, dev, at):
    """A bias that starts at any element of a buffer (a view into flat
    parameters), as the conv takes it: the same bits as an aligned copy."""
    import torch

    print(f"[case] products conv bias at element {at}", flush=True)
    nat = spc._native
    x, w, b, idx = _setup(100, 300, 64, 64, torch.bfloat16, at)
    flat = torch.zeros(64 + 8, dtype=torch.bfloat16, device=dev)
    flat[at:at + 64] = b
    view = flat[at:at + 64]
    assert view.data_ptr() % 8 == 2 * at
    pw = nat.pack_weights(w)
    y = nat.sparse_conv_products(x, pw, view, idx.reshape(-1), n_out=300)
    assert torch.equal(y, nat.sparse_conv_products(x, pw, b, idx.reshape(-1), n_out=300))


def test_products_conv_refuses_what_the_conv_refuses(spc, dev):
    """A negative or NaN eps, residual_rows into no rows and a norm over other
    widths raise, as in sparse_conv."""
    import torch

    nat = spc._native
    x, w, b, idx = _setup(50, 80, 64, 64, torch.bfloat16, 1)
    pw, coords = nat.pack_weights(w), torch.zeros((80, 4), dtype=torch.int32, device=dev)
    mod = torch.zeros((1, 64), device=dev)
    calls = [lambda f, **k: f(norm_mod=(mod, mod, coords, -1.0), **k),
             lambda f, **k: f(norm_mod=(mod, mod, coords, float("nan")), **k)]
    both = [lambda **e: nat.sparse_conv_products(x, pw, b, idx.reshape(-1), n_out=80, **e),
            lambda **e: nat.sparse_conv(x, pw, b, idx.reshape(-1), ntaps=27, n_out=80, **e)]
    for f in both:
        for call in calls:
            print("[case] products conv eps", flush=True)
            with pytest.raises(nat.SparseConvError):
                call(f)
    # the C entries: residual_rows with n_residual 0, and cout 96 with the norm
    L, s = nat.lib(), torch.cuda.current_stream().cuda_stream
    y = torch.empty((80, 64), dtype=torch.bfloat16, device=dev)
    rows = torch.zeros(80, dtype=torch.int32, device=dev)
    ws = torch.empty(L.spc_conv_products_workspace_bytes(50, 64), dtype=torch.uint8, device=dev)
    epi = nat.ConvEpilogue(nat.EPI_RESIDUAL, 0.0, y.data_ptr(), None, None, None, 0,
                           rows.data_ptr(), 0)
    st = L.spc_sparse_conv_products(s, nat.BF16, x.data_ptr(), pw.data.data_ptr(), None,
                                    y.data_ptr(), idx.data_ptr(), 80, 50, 64, 64,
                                    ctypes.byref(epi), ws.data_ptr(), ws.numel())
    assert st == nat.BAD_ARG
    p96 = nat.pack_weights(torch.zeros((96, 27, 64), dtype=torch.bfloat16, device=dev))
    m96 = torch.zeros((1, 96), device=dev)
    codes = []
    for f in (lambda **e: nat.sparse_conv_products(x, p96, None, idx.reshape(-1), n_out=80, **e),
              lambda **e: nat.sparse_conv(x, p96, None, idx.reshape(-1), ntaps=27, n_out=80, **e)):
        with pytest.raises(nat.SparseConvError) as err:
            f(norm_mod=(m96, m96, coords, 1e-6))
        codes.append(err.value.status)
    assert codes[0] == codes[1]


def test_products_conv_equals_conv_on_an_upsampled_level(spc, dev):
    """The up block's route: the same block with the implicit GEMM agrees to
    the F32 order (a rounding step of the 16-bit intermediates at most), and
    narrow, quantised and f32 convs keep the implicit GEMM."""
    import torch

    sp = spc.sparse
    c = torch.from_numpy(spc.workloads.sphere_shell(32, 12.0)).to(dev)
    ct = sp.SparseDownsample(2)(sp.SparseTensor(torch.zeros((c.shape[0], 32), dtype=torch.bfloat16,
                                                            device=dev), c))
    n_f, n_c = c.shape[0], ct.coords.shape[0]
    print(f"[case] up block by products {n_c} -> {n_f} rows", flush=True)
    torch.manual_seed(5)
    blk = spc.blocks.SparseResBlock3d(256, 64, 128, upsample=True).to(dev).bfloat16()
    blk.norm1.float()
    with torch.no_grad():
        blk.conv2.conv.weight.normal_(0, 0.02)
        x = ct.replace(torch.randn((n_c, 256), device=dev).bfloat16())
        emb = torch.randn((1, 64), device=dev).bfloat16()
        assert blk.conv1._use_products(torch.bfloat16, n_f, n_c)
        y = blk(x, emb).feats.float()
        blk.conv1._use_products = lambda *a: False
        y0 = blk(x, emb).feats.float()
    assert float((y - y0).norm() / y0.norm()) <= 2.0 ** -8
    k = sp.SparseConv3d(256, 128, 3)
    assert not k._use_products(torch.float32, n_f, n_c)
    assert not k._use_products(torch.bfloat16, 2 * n_c, n_c)
    assert not sp.SparseConv3d(128, 128, 3)._use_products(torch.bfloat16, n_f, n_c)


def test_up_block_runs_without_room_for_the_products(spc, dev, monkeypatch):
    """Where the products' buffer cannot be allocated the up block runs the
    implicit GEMM, with its bits."""
    import torch

    sp, nat = spc.sparse, spc._native
    c = torch.from_numpy(spc.workloads.sphere_shell(32, 12.0)).to(dev)
    ct = sp.SparseDownsample(2)(sp.SparseTensor(torch.zeros((c.shape[0], 32), dtype=torch.bfloat16,
                                                            device=dev), c))
    n_c = ct.coords.shape[0]
    print(f"[case] up block without the products' buffer {n_c} -> {c.shape[0]} rows", flush=True)
    torch.manual_seed(6)
    blk = spc.blocks.SparseResBlock3d(512, 64, 128, upsample=True).to(dev).bfloat16()
    blk.norm1.float()
    x = ct.replace(torch.randn((n_c, 512), device=dev).bfloat16())
    emb = torch.randn((1, 64), device=dev).bfloat16()
    room, need = nat._workspace, 27 * 4 * n_c * 128

    def full(nbytes, device):
        if nbytes >= need:
            raise torch.OutOfMemoryError("no room")
        return room(nbytes, device)

    with torch.no_grad():
        blk.conv2.conv.weight.normal_(0, 0.02)
        assert blk.conv1._use_products(torch.bfloat16, c.shape[0], n_c)
        monkeypatch.setattr(nat, "_workspace", full)
        y = blk(x, emb).feats
        monkeypatch.setattr(nat, "_workspace", room)
        blk.conv1._use_products = lambda *a: False
        assert torch.equal(y, blk(x, emb).feats)
