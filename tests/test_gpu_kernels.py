"""HIP kernels vs the CPU oracle on identical seeded inputs (GPU only).

Each drop-in function is compared with the oracle's restatement of the
reference's torch branch (oracle/schedule.py); the whole schedule is compared
with the fp64 oracle.  Tolerances:
  * fp32 inputs: max|got - ref| / max|ref| < 1e-5 against fp64 on the same values
    (the bar stated for fp32), except where noted;
  * bf16 inputs: O within 2e-2 absolute and log-normaliser within 1e-3
    absolute of the reference torch path (the bar stated for bf16);
  * pooled tables / chunk summaries from bf16 inputs are exact products summed
    in fp32, so they are held to 1e-5 relative against fp64 as well.
"""
import contextlib
import math

import pytest
import torch

import oracle.schedule as O
from smat_attention_amd import attention as A
from smat_attention_amd.kernels import hip_fwd as K
from smat_attention_amd.kernels._lib import general_kernel
from smat_attention_amd.mask import build_mask

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _say(*a):
    print("[case]", *a, flush=True)


def _rel(got, ref):
    got, ref = got.double().cpu(), ref.double().cpu()
    return ((got - ref).abs().max() / ref.abs().max().clamp_min(1e-300)).item()


def _feats(nb, T, hd, dt, seed=0, k_scale=1.0, q_scale=1.0, v_scale=1.0, r=None):
    r = r or hd
    Q, Kk, V = O.seeded_qkv(nb, T, hd, hd, seed=seed, dtype=torch.float32,
                            q_scale=q_scale, k_scale=k_scale, v_scale=v_scale)
    phi = O.make_phi(hd, r, dtype=torch.float32, seed=0)
    Phi, Psi, Vb = O.featurise(Q, Kk, V, phi)
    return Phi.to(dt), Psi.to(dt), Vb.to(dt)


# ---------------------------------------------------------------------------
# drop-in kernels
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("C,r,p", [(128, 128, 129), (128, 64, 65), (64, 32, 33), (256, 64, 65)])
def test_chunk_local(dt, C, r, p):
    _say("chunk_local", dt, C, r, p)
    nb, nc = 2, 3
    g = torch.Generator().manual_seed(1)
    Phi = (torch.rand(nb, nc, C, r, generator=g) + 0.5).to(dt)
    Psi = (torch.rand(nb, nc, C, r, generator=g) + 0.5).to(dt)
    Vb = torch.randn(nb, nc, C, p, generator=g).to(dt)
    Sin = torch.randn(nb, nc, r, p, generator=g) * 10
    got = K.chunk_local(Phi.to(DEV), Psi.to(DEV), Vb.to(DEV), Sin.to(DEV))
    torch.cuda.synchronize()
    assert got.dtype == torch.float32 and got.shape == (nb, nc, C, p)
    if dt == torch.float32:
        ref = O.chunk_local(Phi.double(), Psi.double(), Vb.double(), Sin.double())
        assert _rel(got, ref) < 1e-5
    else:
        # the reference's own path: score tile rounded to the input dtype
        ref = O.chunk_local(Phi, Psi, Vb, Sin, torch.float32)
        assert _rel(got, ref) < 1e-2
        # and the exact product on the same inputs, up to that rounding
        ref64 = O.chunk_local(Phi.double(), Psi.double(), Vb.double(), Sin.double())
        assert _rel(got, ref64) < 3e-2


def test_chunk_local_ragged_and_strided_vb():
    _say("chunk_local ragged C=100, padded Vb rows")
    nb, nc, C, r, p = 2, 2, 100, 64, 65
    g = torch.Generator().manual_seed(2)
    Phi = torch.rand(nb, nc, C, r, generator=g) + 0.5
    Psi = torch.rand(nb, nc, C, r, generator=g) + 0.5
    Vb = torch.randn(nb, nc, C, p, generator=g)
    Sin = torch.randn(nb, nc, r, p, generator=g)
    buf = torch.zeros(nb, nc, C, 72, device=DEV)
    buf[..., :p] = Vb.to(DEV)
    got = K.chunk_local(Phi.to(DEV), Psi.to(DEV), buf[..., :p], Sin.to(DEV))
    ref = O.chunk_local(Phi.double(), Psi.double(), Vb.double(), Sin.double())
    assert _rel(got, ref) < 1e-5


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,d,n_P", [(4096, 2, 0), (4096, 3, 0), (8192, 3, 0), (2048, 3, 16),
                                     (4096, 1, 0)])
def test_pool(dt, T, d, n_P):
    _say("pool", dt, T, d, n_P)
    spec = build_mask(T, d, chunk=128, n_P=n_P)
    Phi, Psi, Vb = _feats(2, T, 32, dt, seed=3)
    Fg = torch.empty(2, 32, 33, device=DEV) if n_P else None
    F = K.pool(Psi.to(DEV), Vb.to(DEV), spec.n_P, spec.n, spec.N0, F_glob=Fg)
    ref = O.pool_profiles(Psi.double(), Vb.double(), spec)
    assert F.shape == ref.shape and F.dtype == torch.float32
    assert _rel(F, ref) < 1e-5
    if n_P:
        gref = Psi[:, :n_P].double().transpose(-1, -2) @ Vb[:, :n_P].double()
        assert _rel(Fg, gref) < 1e-5
    assert K.pool_ok(spec.N0, -(-(spec.n - spec.n_P) // spec.N0), 33)


@pytest.mark.parametrize("T,d", [(4096, 2), (4096, 3), (8192, 4), (1024, 3)])
def test_incidence(T, d):
    _say("incidence", T, d)
    spec = A.to_device(build_mask(T, d, chunk=128), DEV)
    g = torch.Generator().manual_seed(4)
    F = torch.randn(2, spec.N0, 32, 33, generator=g)
    U = K.incidence(F.to(DEV), spec.plane_pts_t, spec.B)
    ref = O.apply_incidence(F.double(), spec)
    assert _rel(U, ref) < 1e-6
    # the schedule-level wrapper reads the parity-interleaved int32 table: the
    # same points per row, summed in another order
    U2 = A.apply_incidence(F.to(DEV), spec)
    assert _rel(U2, ref) < 1e-6


@pytest.mark.parametrize("T,n_P,rp,glob", [
    (2048, 0, (32, 33), True), (32768, 0, (128, 129), True), (131072, 0, (128, 129), True),
    (2048, 16, (32, 33), True), (131072, 0, (128, 129), False), (1024, 0, (8, 9), False),
    (512, 0, (4, 7), True)])
def test_incidence_generated_lines(T, n_P, rp, glob):
    # r*p = 72 and 28 leave a partial last 16-float slice
    _say("incidence, d=3 lines generated in-kernel", T, n_P, rp, glob)
    spec = A.to_device(build_mask(T, 3, chunk=128 if T >= 2048 else 64, n_P=n_P), DEV)
    assert spec.plane_code_t is not None
    g = torch.Generator().manual_seed(8)
    r, p = rp
    nb = 1 if T >= 32768 else 2
    F = torch.randn(nb, spec.N0, r, p, generator=g)
    Fg = torch.randn(nb, r, p, generator=g)
    U = K.incidence_plane(F.to(DEV), spec.plane_code_t, spec.q,
                          F_glob=Fg.to(DEV) if glob else None)
    ref = O.apply_incidence(F.double(), spec)
    if glob:
        ref = ref + Fg.double().unsqueeze(1)
    assert _rel(U, ref) < 1e-6


@pytest.mark.parametrize("T,chunk,q", [(64, 32, 5), (256, 32, 7), (768, 32, 11), (3072, 32, 13),
                                     (6144, 32, 17), (12288, 32, 19), (16384, 32, 23),
                                     (24576, 32, 29), (49152, 32, 31), (65536, 32, 37),
                                     (131072, 32, 41)])
@pytest.mark.parametrize("glob", [False, True])
def test_incidence_line_groups_every_field(T, chunk, q, glob):
    """The line-group kernel is compiled once per prime q: each instantiation the
    masks reach against the fp64 oracle, at r*p = 20 (one whole and one partial
    16-float slice), with and without the global channel."""
    _say("incidence line groups", T, chunk, q, glob)
    spec = A.to_device(build_mask(T, 3, chunk=chunk), DEV)
    assert spec.q == q and spec.plane_code_t is not None
    g = torch.Generator().manual_seed(q)
    F = torch.randn(2, spec.N0, 4, 5, generator=g)
    Fg = torch.randn(2, 4, 5, generator=g)
    U = K.incidence_plane(F.to(DEV), spec.plane_code_t, spec.q,
                          F_glob=Fg.to(DEV) if glob else None)
    ref = O.apply_incidence(F.double(), spec)
    if glob:
        ref = ref + Fg.double().unsqueeze(1)
    assert _rel(U, ref) < 1e-6


@pytest.mark.parametrize("T,chunk,q", [(139264, 32, 43), (163840, 32, 47), (229376, 32, 53),
                                     (327680, 32, 59), (425984, 32, 61), (458752, 32, 67),
                                     (655360, 32, 71), (720896, 32, 73), (786432, 32, 79),
                                     (1048576, 32, 83)])
@pytest.mark.parametrize("glob", [False, True])
def test_incidence_row_groups_every_field(T, chunk, q, glob):
    """The row-group kernel (one plane an item, a line group per sixteen-lane
    row) takes the primes 43 .. 83: each instantiation against the fp64 oracle at
    r*p = 20 (five planes), with and without the global channel."""
    _say("incidence row groups", T, chunk, q, glob)
    spec = A.to_device(build_mask(T, 3, chunk=chunk), DEV)
    assert spec.q == q and spec.plane_code_t is not None
    g = torch.Generator().manual_seed(q)
    F = torch.randn(3, spec.N0, 4, 5, generator=g)
    Fg = torch.randn(3, 4, 5, generator=g)
    U = K.incidence_plane(F.to(DEV), spec.plane_code_t, spec.q,
                          F_glob=Fg.to(DEV) if glob else None)
    ref = O.apply_incidence(F.double(), spec)
    if glob:
        ref = ref + Fg.double().unsqueeze(1)
    assert _rel(U, ref) < 1e-6


@pytest.mark.parametrize("T,q,glob", [(139264, 43, True), (458752, 67, False)])
def test_incidence_row_groups_many_items(T, q, glob):
    """r*p = 1056 over two sequences: 528 one-plane items, several a workgroup,
    so the register prefetch of the next item is exercised."""
    _say("incidence row groups, several items a workgroup", T, q, glob)
    spec = A.to_device(build_mask(T, 3, chunk=32), DEV)
    assert spec.q == q
    g = torch.Generator().manual_seed(T)
    F = torch.randn(2, spec.N0, 32, 33, generator=g)
    Fg = torch.randn(2, 32, 33, generator=g)
    U = K.incidence_plane(F.to(DEV), spec.plane_code_t, spec.q,
                          F_glob=Fg.to(DEV) if glob else None)
    ref = O.apply_incidence(F.double(), spec)
    if glob:
        ref = ref + Fg.double().unsqueeze(1)
    assert _rel(U, ref) < 1e-6


def test_incidence_ragged_endpoint_csr():
    _say("incidence ragged (endpoint mask, CSR)")
    spec = A.to_device(build_mask(256, 8, chunk=8), DEV)
    assert spec.kind == "endpoint" and not spec.uniform_deg
    g = torch.Generator().manual_seed(5)
    F = torch.randn(2, spec.N0, 16, 17, generator=g)
    U = A.apply_incidence(F.to(DEV), spec)
    ref = O.apply_incidence_csr(F.double(), spec)
    assert _rel(U, ref) < 1e-6


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,d,r,p", [(4096, 3, 32, 33), (8192, 2, 64, 65), (4096, 3, 80, 65),
                                     (4096, 3, 96, 80), (4096, 1, 128, 129),
                                     (32768, 3, 128, 129), (131072, 3, 128, 129)])
def test_query(dt, T, d, r, p):
    _say("query", dt, T, d, r, p)
    spec = build_mask(T, d, chunk=128)
    g = torch.Generator().manual_seed(6)
    Phi = (torch.rand(2, spec.T_R, r, generator=g) + 0.5).to(dt)
    U = torch.randn(2, spec.B, r, p, generator=g)
    Y = K.query(Phi.to(DEV), U.to(DEV))
    ref = O.query_by_type(Phi.double(), U.double(), spec)
    # 16-bit Phi is exact; U enters as hi + lo 16-bit parts (~2^-16 relative)
    assert _rel(Y, ref) < (1e-5 if dt == torch.float32 else 2e-5)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T_R", [(300, 300 * 48), (300, 300 * 48 + 1), (300, 300 * 64),
                                   (257, 257 * 57 + 130), (1, 40)])
def test_query_streaming_rows_per_type(dt, B, T_R):
    """The streaming query (16-bit Phi, r = 128, p = 129) at the edges of its
    two tile counts: three 16-row tiles up to 48 rows a type, four up to 64
    (49 rows for the first type only, 57-58 as at T = 524288, d = 3), and a
    single type; against fp64 (U enters as hi + lo 16-bit parts)."""
    from types import SimpleNamespace
    _say("query streaming rows per type", dt, B, T_R)
    g = torch.Generator().manual_seed(17)
    nb = 2
    Phi = (torch.rand(nb, T_R, 128, generator=g) + 0.5).to(dt)
    U = torch.randn(nb, B, 128, 129, generator=g)
    Y = K.query(Phi.to(DEV), U.to(DEV))
    ref = O.query_by_type(Phi.double(), U.double(), SimpleNamespace(B=B))
    assert _rel(Y, ref) < 2e-5


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,d,n_P", [(4096, 3, 0), (8192, 2, 0), (2048, 3, 16), (32768, 3, 0),
                                     (32768, 2, 0), (32768, 2, 16)])
def test_pool_streaming_head_dim_128(dt, T, d, n_P):
    """The DMA-streamed Gram kernel (16-bit, r = 128, p = 129) on the profile
    pool, incl. the global channel, against fp64 and the general kernel.
    Profiles of at most 64 tokens take its single-buffer form; d = 2 at
    T = 32768 (about 125 tokens a profile) the double-buffered one."""
    _say("pool streaming", dt, T, d, n_P)
    spec = build_mask(T, d, chunk=128, n_P=n_P)
    nb = 4
    Phi, Psi, Vb = _feats(nb, T, 128, dt, seed=31)
    Vp = torch.zeros(nb, T, 136, dtype=dt)
    Vp[..., :129] = Vb
    Sd, Vd = Psi.to(DEV), Vp.to(DEV)[..., :129]
    Fg = torch.empty(nb, 128, 129, device=DEV) if n_P else None
    F = K.pool(Sd, Vd, spec.n_P, spec.n, spec.N0, F_glob=Fg)
    Fg_old = torch.empty(nb, 128, 129, device=DEV) if n_P else None
    with general_kernel("gram"):
        F_old = K.pool(Sd, Vd, spec.n_P, spec.n, spec.N0, F_glob=Fg_old)
    ref = O.pool_profiles(Psi.double(), Vb.double(), spec)
    assert _rel(F, ref) < 1e-5 and _rel(F_old, ref) < 1e-5
    if n_P:
        gref = Psi[:, :n_P].double().transpose(-1, -2) @ Vb[:, :n_P].double()
        assert _rel(Fg, gref) < 1e-5


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,d,n_P", [(8192, 3, 0), (8192, 3, 16), (4096, 2, 0)])
def test_pool_head_dim_64_many_profiles(dt, T, d, n_P):
    """The 16-bit r = 64, p = 65 Gram kernel (taken when a launch has at least
    512 items) on the profile pool, incl. the global channel's last-item
    buffer, Vb rows 72 apart as featurise lays them out: against fp64 and
    against the general kernel on the same inputs."""
    _say("pool head_dim 64", dt, T, d, n_P)
    spec = build_mask(T, d, chunk=128, n_P=n_P)
    nb = 16
    Phi, Psi, Vb = _feats(nb, T, 64, dt, seed=37)
    Vp = torch.zeros(nb, T, 72, dtype=dt)
    Vp[..., :65] = Vb
    Sd, Vd = Psi.to(DEV), Vp.to(DEV)[..., :65]
    assert nb * spec.N0 >= 512
    Fg = torch.empty(nb, 64, 65, device=DEV) if n_P else None
    F = K.pool(Sd, Vd, spec.n_P, spec.n, spec.N0, F_glob=Fg)
    Fg_old = torch.empty(nb, 64, 65, device=DEV) if n_P else None
    with general_kernel("gram"):
        F_old = K.pool(Sd, Vd, spec.n_P, spec.n, spec.N0, F_glob=Fg_old)
    ref = O.pool_profiles(Psi.double(), Vb.double(), spec)
    assert _rel(F, ref) < 1e-5 and _rel(F_old, ref) < 1e-5
    if n_P:
        gref = Psi[:, :n_P].double().transpose(-1, -2) @ Vb[:, :n_P].double()
        assert _rel(Fg, gref) < 1e-5 and _rel(Fg_old, gref) < 1e-5


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_chunk_states_and_segment_scan(dt):
    _say("chunk_states + segment_scan", dt)
    nb, T, C, r, p, n = 2, 2048 + 77, 128, 64, 65, 1024
    Phi, Psi, Vb = _feats(nb, T, 64, dt, seed=7)
    D = K.chunk_states(Psi.to(DEV), Vb.to(DEV), C)
    pad = (-T) % C
    Psi_p = torch.nn.functional.pad(Psi.double(), (0, 0, 0, pad))
    Vb_p = torch.nn.functional.pad(Vb.double(), (0, 0, 0, pad))
    nc = (T + pad) // C
    Dref, Sref = O.chunk_states(Psi_p.reshape(nb, nc, C, r), Vb_p.reshape(nb, nc, C, p), n, C,
                                torch.float64)
    assert _rel(D, Dref) < 1e-5
    Sin = K.segment_scan(D, n // C)
    assert _rel(Sin, Sref) < 1e-5
    # the reset: the first chunk of each segment sees a zero state, exactly
    assert torch.count_nonzero(Sin[:, 0]).item() == 0
    assert torch.count_nonzero(Sin[:, n // C]).item() == 0


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("vb_pad", [False, True])
def test_chunk_states_many_sequences(dt, vb_pad):
    """The 16-bit r = 64, p = 65 chunk-summary kernel (taken when a launch has
    at least 512 items): 64 sequences, a ragged last chunk, Vb rows 65 or 72
    apart, against fp64 sums of the same values; and the causal pass that
    uses it for its group summaries (two chunks a group at this size, split
    at n) against the oracle's scan."""
    _say("chunk_states many sequences", dt, vb_pad)
    nb, T, C, r, p, n = 64, 3000, 128, 64, 65, 1024
    Phi, Psi, Vb = _feats(nb, T, 64, dt, seed=17)
    Vd = Vb.to(DEV)
    if vb_pad:
        Vp = torch.zeros(nb, T, 72, dtype=dt, device=DEV)
        Vp[..., :p] = Vd
        Vd = Vp[..., :p]
    D = K.chunk_states(Psi.to(DEV), Vd, C)
    pad = (-T) % C
    nc = (T + pad) // C
    Psi_p = torch.nn.functional.pad(Psi.double(), (0, 0, 0, pad))
    Vb_p = torch.nn.functional.pad(Vb.double(), (0, 0, 0, pad))
    Dref = torch.einsum("bcta,bctv->bcav", Psi_p.reshape(nb, nc, C, r),
                        Vb_p.reshape(nb, nc, C, p))
    assert _rel(D, Dref) < 1e-5
    H = K.causal_scan(Phi.to(DEV), Psi.to(DEV), Vd, n, C, write_H=True)
    ref = O.segmented_causal_scan(Phi[:4], Psi[:4], Vb[:4], n, chunk=C)
    assert _rel(H[:4], ref) < 1e-2


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,n,C,hd", [(2048, 1024, 128, 64), (2048 + 77, 1024, 128, 32),
                                      (4096, 2048, 64, 32), (1000, 0, 128, 32),
                                      (8192, 4096, 128, 128), (300, 256, 128, 16),
                                      (2048 + 40, 1024, 64, 48)])
def test_causal_scan_fused(dt, T, n, C, hd):
    _say("causal scan fused", dt, T, n, C, hd)
    Phi, Psi, Vb = _feats(2, T, hd, dt, seed=9)
    H = K.causal_scan(Phi.to(DEV), Psi.to(DEV), Vb.to(DEV), n, C, write_H=True)
    if dt == torch.float32:
        ref = O.segmented_causal_scan(Phi.double(), Psi.double(), Vb.double(), n, chunk=C)
        assert _rel(H, ref) < 1e-5
    else:
        ref = O.segmented_causal_scan(Phi, Psi, Vb, n, chunk=C)
        assert _rel(H, ref) < 1e-2
    # normalised mode with a long-range term on the recent rows and a gate
    g = torch.Generator().manual_seed(10)
    Y = torch.rand(2, T - n, Vb.shape[-1], generator=g)
    gate = torch.rand(2, T, generator=g) + 0.5
    out = K.causal_scan(Phi.to(DEV), Psi.to(DEV), Vb.to(DEV), n, C, Y=Y.to(DEV), g=gate.to(DEV))
    Hr = ref.double().clone()
    Hr[:, n:] += Y.double()
    want = Hr[..., :-1] / Hr[..., -1:] * gate.double().unsqueeze(-1)
    tol = 1e-5 if dt == torch.float32 else 2e-2
    assert (out.double().cpu() - want).abs().max().item() < tol * max(1.0, want.abs().max().item())


@pytest.mark.parametrize("nb,T,n,C,r", [(8, 32768, 16384, 8, 8), (4, 4096, 56, 8, 72),
                                        (3, 4096 + 5, 2048, 8, 72), (1, 64, 64, 8, 72),
                                        (5, 2049, 0, 8, 8)])
def test_causal_scan_group_sizes(nb, T, n, C, r):
    """The causal pass with many chunks a group (both tile shapes), groups cut
    short by n and by T, and n far from the half the grouping assumes, against
    fp64."""
    _say("causal scan groups", nb, T, n, C, r)
    Phi, Psi, Vb = _feats(nb, T, r, torch.float32, seed=33)
    H = K.causal_scan(Phi.to(DEV), Psi.to(DEV), Vb.to(DEV), n, C, write_H=True)
    ref = O.segmented_causal_scan(Phi.double(), Psi.double(), Vb.double(), n, chunk=C)
    assert _rel(H, ref) < 1e-5


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,n,C", [(4096, 2048, 128), (8192, 0, 128), (4096, 4096, 128),
                                   (4096, 1024, 64), (2048 + 64, 1024, 128), (16384, 8192, 128)])
def test_causal_scan_streaming(dt, T, n, C):
    """The head_dim-128 streaming kernel (16-bit inputs, p = 129, 64-token
    steps through LDS) against the oracle's reference path, and against the
    general fused kernel on the same inputs."""
    _say("causal scan streaming", dt, T, n, C)
    hd = 128
    Phi, Psi, Vb = _feats(2, T, hd, dt, seed=21)
    P = Vb.shape[-1]
    g = torch.Generator().manual_seed(22)
    Y = torch.rand(2, T - n, P, generator=g)
    gate = torch.rand(2, T, generator=g) + 0.5
    # Vb rows padded to 136 and Y rows to 132, as featurise / query lay them out
    Vp = torch.zeros(2, T, 136, dtype=dt)
    Vp[..., :P] = Vb
    Yp = torch.zeros(2, T - n, 132)
    Yp[..., :P] = Y
    Pd, Sd = Phi.to(DEV), Psi.to(DEV)
    Vd = Vp.to(DEV)[..., :P]
    Yd = Yp.to(DEV)[..., :P] if T > n else None
    gd = gate.to(DEV)
    out = K.causal_scan(Pd, Sd, Vd, n, C, Y=Yd, g=gd)
    with general_kernel("scan"):
        old = K.causal_scan(Pd, Sd, Vd, n, C, Y=Yd, g=gd)
    torch.cuda.synchronize()
    ref = O.segmented_causal_scan(Phi, Psi, Vb, n, chunk=C).double()
    if T > n:
        ref[:, n:] += Y.double()
    want = ref[..., :-1] / ref[..., -1:] * gate.double().unsqueeze(-1)
    scale = max(1.0, want.abs().max().item())
    e_new = (out.double().cpu() - want).abs().max().item() / scale
    e_old = (old.double().cpu() - want).abs().max().item() / scale
    _say(f"  streaming {e_new:.2e}  fused {e_old:.2e}")
    assert torch.isfinite(out).all()
    assert e_new < 2e-2 and e_old < 2e-2
    # the streaming kernel rounds scores per 64-token step, the fused kernel
    # per chunk: close, not identical -- so the two paths really both ran
    assert not torch.equal(out, old)
    assert (out - old).abs().max().item() / scale < 1e-2


# ---------------------------------------------------------------------------
# the whole schedule
# ---------------------------------------------------------------------------

def _check_forward(spec, Phi, Psi, Vb, *, dt, g=None, label=""):
    Pd, Sd, Wd = (x.to(DEV) for x in (Phi, Psi, Vb))
    gd = g.to(DEV) if g is not None else None
    out, parts = A.smat_attention(Pd, Sd, Wd, spec, g=gd, return_parts=True)
    fused = A.smat_attention(Pd, Sd, Wd, spec, g=gd)
    torch.cuda.synchronize()
    ref64, p64 = O.smat_attention(Phi.double(), Psi.double(), Vb.double(), spec, g=g,
                                  return_parts=True)
    lse = torch.log(parts["H"][..., -1].double().cpu())
    lse64 = torch.log(p64["H"][..., -1])
    e_fused = (fused - out).abs().max().item()
    if dt == torch.float32:
        rel = _rel(out, ref64)
        _say(label, f"fp32 rel {rel:.2e}, lse {((lse - lse64).abs().max().item()):.2e}")
        assert rel < 1e-5
        assert (lse - lse64).abs().max().item() < 1e-5
    else:
        refbf, pbf = O.smat_attention(Phi, Psi, Vb, spec, g=g, return_parts=True)
        lsebf = torch.log(pbf["H"][..., -1].double())
        e_o = (out.double().cpu() - refbf.double()).abs().max().item()
        e_l = (lse - lsebf).abs().max().item()
        e_o64 = (out.double().cpu() - ref64).abs().max().item()
        e_l64 = (lse - lse64).abs().max().item()
        _say(label, f"vs torch path: O {e_o:.2e} lse {e_l:.2e}; vs fp64: O {e_o64:.2e} "
                    f"lse {e_l64:.2e}")
        # the bar: the reference's torch path on the same bf16 inputs
        assert e_o < 2e-2 and e_l < 1e-3
        # the exact schedule on the same values differs by the reference's own
        # rounding of the score tile to bf16 (up to 2^-8 on a one-term row)
        assert e_o64 < 2e-2 and e_l64 < 1e-2
    assert e_fused <= 1e-6 * max(1.0, out.abs().max().item())
    return out


@pytest.mark.parametrize("dt,nb,T,n,hd,K", [
    (torch.bfloat16, 96, 1024, 512, 80, 1), (torch.float32, 96, 1024, 512, 128, 1),
    (torch.float32, 24, 1024, 512, 128, 1), (torch.bfloat16, 56, 2048, 1024, 72, 2),
    (torch.bfloat16, 48, 4096, 2048, 64, 1), (torch.float32, 96, 4096, 2048, 16, 2),
    (torch.bfloat16, 8, 10007, 4992, 80, 3), (torch.bfloat16, 36, 8913, 4352, 80, 2),
    (torch.float32, 88, 1795, 896, 72, 1)])
def test_causal_scan_general_groups(dt, nb, T, n, hd, K):
    """The general kernel (fp32, and 16-bit value rows that are not 16-byte aligned)
    takes the group of K chunks that measured fastest, not the streaming kernel's
    larger one: the workspace holds the groups of K and the pass stays inside it,
    with its values as in fp64 (a few sequences; 16 bits: scores rounded once)."""
    from smat_attention_amd.kernels.hip_fwd import DTYPE_CODE, _lib, call, stream_of
    _say("causal scan general groups", dt, nb, T, n, hd, K)
    P, nc = hd + 1, -(-T // 128)
    Phi, Psi, Vb = (t.to(DEV) for t in _feats(nb, T, hd, dt, seed=91))
    wsb = _lib.query("smat_causal_scan_workspace_bytes", nb, T, 128, hd, P)
    assert wsb >= 2 * nb * (-(-nc // K)) * hd * P * 4
    ws = torch.full((wsb + 512,), 0x5A, device=DEV, dtype=torch.uint8)
    off = -ws.data_ptr() % 256
    H = torch.empty(nb, T, P, device=DEV)
    call("smat_causal_scan", DTYPE_CODE[dt], Phi.data_ptr(), Psi.data_ptr(), Vb.data_ptr(), 0, 0,
         H.data_ptr(), nb, T, n, 128, hd, P, T * hd, hd, T * hd, hd, T * P, P, 0, 0, T * P, P, 0, 1,
         ws.data_ptr() + off, wsb, stream_of(H))
    assert (ws[:off] == 0x5A).all() and (ws[off + wsb:] == 0x5A).all()
    some = [0, nb // 2, nb - 1]
    ref = O.segmented_causal_scan(*(t[some].double().cpu() for t in (Phi, Psi, Vb)), n, chunk=128)
    assert _rel(H[some], ref) < (1e-5 if dt == torch.float32 else 2.0 ** -8)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nb,T,n,hd", [(64, 600, 256, 16), (31, 1000, 512, 16), (63, 130, 128, 64),
                                       (128, 256, 128, 64), (1, 127, 0, 64), (2, 4096, 2048, 64)])
def test_causal_scan_small_batches(dt, nb, T, n, hd):
    """The causal pass at chunk 128 on both sides of the line under which it runs
    halved chunks (fewer than 256 of them; 31 x 8 halves once, 64 x 5 not at all),
    short last chunks included, against fp64 (scores rounded once in 16 bits)."""
    _say("causal scan small batches", dt, nb, T, n, hd)
    Phi, Psi, Vb = _feats(nb, T, hd, dt, seed=71)
    Vp = torch.zeros(nb, T, hd + 8, dtype=dt)
    Vp[..., :hd + 1] = Vb
    H = K.causal_scan(Phi.to(DEV), Psi.to(DEV), Vp.to(DEV)[..., :hd + 1], n, 128, write_H=True)
    ref = O.segmented_causal_scan(Phi.double(), Psi.double(), Vb.double(), n, chunk=128)
    assert _rel(H, ref) < (1e-5 if dt == torch.float32 else 2.0 ** -8)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hd,stride", [(32, 40), (40, 48), (64, 65), (64, 72), (128, 129),
                                       (128, 136)])
def test_causal_scan_of_one_sequence_and_of_a_batch(hd, stride, dt):
    """A sequence gives the same rows alone, among 64 (more than 256 chunks) and, up to
    its length, in a longer one: in 16 bits the same scores are rounded whatever the
    call's size, on the general kernel (narrow heads, value rows that are not
    16-byte aligned) and the streaming one; what may differ is the order of the
    states' fp32 sums."""
    _say("causal scan, one and a batch", hd, stride, dt)
    nb, T, n = 64, 1024, 512
    gen = torch.Generator().manual_seed(81)
    Phi, Psi = (torch.rand(nb, T, hd, generator=gen).to(dt).to(DEV) for _ in range(2))
    Vb = torch.randn(nb, T, stride, generator=gen).to(dt).to(DEV)
    Vb[..., hd] = 1.0
    Vb = Vb[..., :hd + 1]
    for wh in (False, True):
        many = K.causal_scan(Phi, Psi, Vb, n, 128, write_H=wh)
        one = K.causal_scan(Phi[:1], Psi[:1], Vb[:1], n, 128, write_H=wh)
        short = K.causal_scan(Phi[:1, :640], Psi[:1, :640], Vb[:1, :640], n, 128, write_H=wh)
        for got, want in ((one, many[:1]), (short, many[:1, :640])):
            assert _rel(got, want) < 2e-6
    spec = A.to_device(build_mask(T, 2, chunk=128), DEV)
    many = A.smat_attention(Phi, Psi, Vb, spec)
    assert _rel(A.smat_attention(Phi[:1], Psi[:1], Vb[:1], spec), many[:1]) < 2e-6


@pytest.mark.parametrize("hd,T", [(64, 1024), (80, 1024), (96, 1000), (112, 1024), (128, 1000)])
def test_causal_scan_fp16_last_states(hd, T):
    """fp16 segments whose state passes 65504 only in their last chunk, which the
    streaming kernel reads there and the general one never forms: both give the
    pass in fp64 (scores rounded once to fp16, 2^-12 each; the states within that)."""
    _say("causal scan, last states of fp16", hd, T)
    nb, n, dt = 2, 512, torch.float16
    gen = torch.Generator().manual_seed(53)
    u = lambda *s: torch.rand(*s, generator=gen)
    Phi, Psi = (2.0 ** -9 + 2.0 ** -7 * u(nb, T, hd)).to(dt), (150 + 10 * u(nb, T, hd)).to(dt)
    for a in (0, n):
        S = Psi[:, a:a + n].double().cumsum(1)
        assert (S[:, 383] < 65504).all() and (S[:, 447] > 65520).all()
    Vb = torch.ones(nb, T, hd + 8, dtype=dt)
    Vb[..., :hd] = torch.randn(nb, T, hd, generator=gen).to(dt)
    ref = O.segmented_causal_scan(Phi.double(), Psi.double(), Vb[..., :hd + 1].double(), n,
                                  chunk=128)
    x = (Phi.to(DEV), Psi.to(DEV), Vb.to(DEV)[..., :hd + 1])
    for which in (general_kernel("scan"), contextlib.nullcontext()):
        with which:
            H = K.causal_scan(*x, n, 128, write_H=True)
            o = K.causal_scan(*x, n, 128, write_H=False)
        for got, want in ((H, ref), (o, ref[..., :-1] / ref[..., -1:])):
            assert torch.isfinite(got).all() and _rel(got, want) < 2.0 ** -10


@pytest.mark.parametrize("gate", [False, True])
@pytest.mark.parametrize("hd", [64, 80, 96, 112, 128])
def test_causal_scan_divides_large_normalisers(hd, gate):
    """bf16 normalisers past 2^126, whose reciprocals are below the smallest normal
    value, and gates times reciprocals that are: the running mean of the values,
    as the general kernel gives it (scores exact; 2^-20 for a subnormal reciprocal)."""
    _say("causal scan, large normalisers", hd, gate)
    T, bf = 31, torch.bfloat16
    Phi = torch.full((1, T, hd), 2.0 ** 58, dtype=bf, device=DEV)
    Vb = torch.ones(1, T, hd + 8, dtype=bf, device=DEV)
    Vb[..., :hd] = torch.rand(1, T, hd, generator=torch.Generator().manual_seed(57)).to(bf)
    Vb = Vb[..., :hd + 1]
    V = Vb[..., :hd].double()
    want = V.cumsum(1) / torch.arange(1, T + 1, device=DEV).view(1, T, 1)
    g = torch.full((1, T), 2.0 ** -30, device=DEV) if gate else None
    for which in (general_kernel("scan"), contextlib.nullcontext()):
        with which:
            o = K.causal_scan(Phi, Phi, Vb, 0, 128, g=g)
        assert _rel(o, want * (2.0 ** -30 if gate else 1.0)) < 2.0 ** -20


@pytest.mark.parametrize("hd", [80, 96, 112])
@pytest.mark.parametrize("T,n_P,n,N0,nb", [(2048, 0, 1024, 121, 3), (2048, 16, 1000, 90, 3),
                                           (9000, 64, 8000, 50, 6), (640, 0, 640, 640, 1)])
def test_gram_streaming_widths(hd, T, n_P, n, N0, nb):
    """The streaming Gram sums between head sizes 64 and 128 (five to seven waves):
    profiles of one step and of several, a short last step, one token a profile,
    the global channel, and chunk groups, from rows whose padding is NaN, against
    fp64."""
    _say("gram widths", hd, T, n_P, n, N0, nb)
    Phi, Psi, Vb = _feats(nb, T, hd, torch.bfloat16, seed=51)
    Vp = torch.full((nb, T, hd + 8), float("nan"), dtype=torch.bfloat16)
    Vp[..., :hd + 1] = Vb
    Sd, Vd = Psi.to(DEV), Vp.to(DEV)[..., :hd + 1]
    glob = torch.empty(nb, hd, hd + 1, device=DEV) if n_P else None
    F = K.pool(Sd, Vd, n_P, n, N0, F_glob=glob)
    S64, V64 = Psi.double(), Vb.double()
    for x in (0, 1, (n - n_P) % N0 - 1, N0 - 1):
        rows = slice(n_P + x % N0, n, N0)
        want = S64[:, rows].transpose(1, 2).contiguous() @ V64[:, rows]
        assert _rel(F[:, x % N0], want) < 1e-5
    if n_P:
        want = S64[:, :n_P].transpose(1, 2).contiguous() @ V64[:, :n_P]
        assert _rel(glob, want) < 1e-5
    C = 64 if nb == 1 else 8
    D = K.chunk_states(Sd, Vd, C)
    pad = torch.nn.functional.pad
    c64 = lambda t: pad(t, (0, 0, 0, -T % C)).reshape(nb, -1, C, t.shape[-1])
    assert _rel(D, c64(S64).transpose(2, 3).contiguous() @ c64(V64)) < 1e-5


@pytest.mark.parametrize("hd", [64, 80, 96, 112])
@pytest.mark.parametrize("T_R,B", [(1024, 47), (300, 132), (1000, 7), (5, 9), (64, 1), (130, 2)])
def test_query_tile_widths(hd, T_R, B):
    """The query between head sizes 64 and 128 (U_h and 64 rows in LDS): several
    row blocks a type, short last blocks, types without a row, against the general
    kernel and fp64 (U split in two 16-bit parts: 2^-15 of the sum of products)."""
    _say("query tile", hd, T_R, B)
    g = torch.Generator().manual_seed(61)
    Phi = (torch.rand(3, T_R, hd, generator=g) + 0.1).to(torch.bfloat16)
    U = torch.randn(3, B, hd, hd + 1, generator=g)
    Pd, Ud = Phi.to(DEV), U.to(DEV)
    got = K.query(Pd, Ud)
    with general_kernel("query"):
        old = K.query(Pd, Ud)
    Ui = U.double()[:, torch.arange(T_R) % B]
    want = (Phi.double().unsqueeze(2) @ Ui).squeeze(2)
    bound = (Phi.double().unsqueeze(2) @ Ui.abs()).squeeze(2) * 2.0 ** -15
    assert ((got.double().cpu() - want).abs() <= bound).all()
    assert _rel(got, old) < 1e-5


@pytest.mark.parametrize("hd,T,n,C,dt", [
    (64, 1024, 512, 128, torch.bfloat16), (64, 64, 0, 64, torch.float16),
    (64, 8192 + 1, 4096, 128, torch.bfloat16), (64, 1023, 1023 // 64 * 64, 64, torch.bfloat16),
    (80, 2048, 1024, 128, torch.float16), (80, 1000, 512, 64, torch.bfloat16),
    (96, 3 * 128 + 17, 128, 128, torch.float16), (96, 2048, 2048, 128, torch.bfloat16),
    (112, 640 + 63, 256, 128, torch.bfloat16), (112, 1024, 0, 128, torch.float16),
    (128, 1000, 512, 128, torch.bfloat16), (128, 65, 64, 64, torch.float16)])
def test_causal_scan_streaming_widths(hd, T, n, C, dt):
    """The streaming scan at every head width it takes (r = 64 .. 128 by 16: four to
    eight waves, an odd k-block of 16 features at 80 and 112) and at lengths that
    are no multiple of its 64-token step: normalised with Y and the gate, with
    neither, and H itself, against the general kernel and the oracle's path."""
    _say("causal scan widths", hd, T, n, C, dt)
    Phi, Psi, Vb = _feats(3, T, hd, dt, seed=41)
    P, pad = hd + 1, hd + 8
    g = torch.Generator().manual_seed(42)
    Y = torch.rand(3, T - n, P, generator=g)
    gate = (torch.rand(3, T, generator=g) + 0.5).to(DEV)
    Vp = torch.full((3, T, pad), float("nan"), dtype=dt)      # the row padding is never data
    Vp[..., :P] = Vb
    Yp = torch.full((3, T - n, (P + 3) // 4 * 4), float("nan"))
    Yp[..., :P] = Y
    Pd, Sd, Vd = Phi.to(DEV), Psi.to(DEV), Vp.to(DEV)[..., :P]
    Yd = Yp.to(DEV)[..., :P] if T > n else None
    runs = (dict(Y=Yd, g=gate), dict(Y=Yd), dict(), dict(write_H=True))
    got = [K.causal_scan(Pd, Sd, Vd, n, C, **kw) for kw in runs]
    with general_kernel("scan"):
        old = [K.causal_scan(Pd, Sd, Vd, n, C, **kw) for kw in runs]
    torch.cuda.synchronize()
    H64 = O.segmented_causal_scan(Phi.double(), Psi.double(), Vb.double(), n, chunk=C)
    Hy = H64.clone()
    if T > n:
        Hy[:, n:] += Y.double()
    norm = lambda H: H[..., :-1] / H[..., -1:]
    want = (norm(Hy) * gate.double().cpu().unsqueeze(-1), norm(Hy), norm(H64), H64)
    for name, a, b, w in zip(("Y, gate", "Y", "plain", "H"), got, old, want):
        scale = w.abs().max().item()
        e_new = (a.double().cpu() - w).abs().max().item() / scale
        e_old = (b.double().cpu() - w).abs().max().item() / scale
        _say(f"  {name}: streaming {e_new:.2e} general {e_old:.2e}")
        assert torch.isfinite(a).all()
        # both round the scores to the input type once; the streaming kernel
        # fewer of them (64-token steps against whole chunks)
        assert e_new <= 1.5 * e_old + 1e-6


def test_forward_plumbing_config_fp32():
    """nb=4 (B=1, H=4), T=1024, d=2, head_dim=64, fp32, q,k,v ~ N(0,1) seed 0."""
    _say("forward T=1024 d=2 nb=4 hd=64 fp32")
    spec = build_mask(1024, 2, chunk=128)
    Phi, Psi, Vb = _feats(4, 1024, 64, torch.float32, seed=0)
    _check_forward(spec, Phi, Psi, Vb, dt=torch.float32, label="T=1024 d=2")
    # and against the O(T^2) definition under the materialised mask
    M = torch.from_numpy(__import__("smat_attention_amd.mask", fromlist=["x"]).materialise(spec))
    dense = O.dense_masked_kernel_attention(Phi.double(), Psi.double(), Vb.double(), M)
    got = A.smat_attention(Phi.to(DEV), Psi.to(DEV), Vb.to(DEV), spec)
    assert _rel(got, dense) < 1e-5


@pytest.mark.parametrize("T,d,n_P", [(2048, 3, 0), (2048, 3, 16), (4096, 4, 0), (2000, 3, 0),
                                     (1024, 1, 0), (4096, 2, 0)])
def test_forward_fp32_small(T, d, n_P):
    _say("forward fp32", T, d, n_P)
    spec = build_mask(T, d, chunk=128, n_P=n_P)
    Phi, Psi, Vb = _feats(2, T, 32, torch.float32, seed=11)
    g = torch.rand(2, T, generator=torch.Generator().manual_seed(12)) + 0.5
    _check_forward(spec, Phi, Psi, Vb, dt=torch.float32, g=g, label=f"T={T} d={d}")


@pytest.mark.parametrize("T,hd,dt,gate", [(1024, 64, torch.float32, True),
                                          (1000, 32, torch.float32, False),
                                          (2048 + 64, 128, torch.bfloat16, False),
                                          (1337, 96, torch.float16, True),
                                          (640, 128, torch.float16, True)])
def test_forward_one_state(T, hd, dt, gate):
    """d = 1: the forward is the causal pass over one segment (every recent row
    reads the state of all landmark tokens); against plain causal attention in
    fp64, scores rounded to the input type as the reference rounds them (ragged
    lengths, the last chunk short; streaming, wide and narrow scans)."""
    _say("forward one state", T, hd, dt, gate)
    spec = build_mask(T, 1, chunk=128)
    Phi, Psi, Vb = _feats(3, T, hd, dt, seed=31)
    g = (torch.rand(3, T, generator=torch.Generator().manual_seed(32)) + 0.5) if gate else None
    got = A.smat_attention(*(x.to(DEV) for x in (Phi, Psi, Vb)), spec,
                           g=None if g is None else g.to(DEV))
    S = Phi.double() @ Psi.double().transpose(1, 2).contiguous()
    H = S.tril() @ Vb.double()
    want = H[..., :-1] / H[..., -1:]
    want = want if g is None else want * g.double().unsqueeze(-1)
    # fp32: the suite's bar; 16-bit: scores rounded to half an ulp (2^-9 bf16,
    # 2^-12 fp16, at most doubled by the division), of values up to max |V|
    tol = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dt]
    e = (got.double().cpu() - want).abs().max().item() / Vb[..., :-1].abs().max().item()
    _say(f"  rel {e:.2e}")
    assert e < tol * (1.5 if gate else 1.0)


@pytest.mark.parametrize("hd,fused", [(32, False), (64, False), (96, False), (128, False),
                                      (128, True)])
def test_forward_d1_fp16_keeps_its_range(hd, fused):
    """d = 1 in fp16, whose states and tables enter the products as hi + lo parts up to
    65504: landmark sums of 51200 and sums of all tokens of 102400 (features near
    100) give the attention of the same values in fp64, scores rounded once to
    fp16 (2^-12 each, at most doubled by the division)."""
    _say("forward d=1 fp16 range", hd, fused)
    T, dt = 1024, torch.float16
    spec = build_mask(T, 1, chunk=128)
    gen = torch.Generator().manual_seed(51)
    u = lambda *s: torch.rand(*s, generator=gen)
    if fused:
        phi = A.FeatureMap(torch.eye(hd, device=DEV, dtype=dt), "elu1")
        Q, Kk, V = ((-7 + 2 * u(2, T, hd)).to(dt), (90 + 20 * u(2, T, hd)).to(dt),
                    torch.randn(2, T, hd, generator=gen).to(dt))
        x = [t.to(DEV) for t in (Q, Kk, V)]
        assert A._fused_ok(*x, phi, spec, 128, None)
        got = A.smat_attention_fused(*x, phi, spec)
        Phi, Psi, Vb = (t.cpu() for t in A.featurise(*x, phi))
    else:
        Phi, Psi = (2.0 ** -9 + 2.0 ** -7 * u(2, T, hd)).to(dt), (90 + 20 * u(2, T, hd)).to(dt)
        Vb = torch.ones(2, T, hd + 8, dtype=dt)
        Vb[..., :hd] = torch.randn(2, T, hd, generator=gen).to(dt)
        Vb = Vb[..., :hd + 1]
        got = A.smat_attention(Phi.to(DEV), Psi.to(DEV),
                               torch.nn.functional.pad(Vb, (0, 7)).to(DEV)[..., :hd + 1], spec)
    S = Phi.double() @ Psi.double().transpose(1, 2).contiguous()
    H = S.tril() @ Vb.double()
    want = H[..., :-1] / H[..., -1:]
    e = (got.double().cpu() - want).abs().max().item() / Vb[..., :-1].abs().max().item()
    _say(f"  rel {e:.2e}")
    assert torch.isfinite(got).all() and e < 2.0 ** -10


def test_forward_single_gpu_d2_bf16():
    """nb=32 (B=4, H=8), T=8192, d=2, head_dim=64, bf16, q,k,v ~ N(0,1)/sqrt(64)."""
    _say("forward T=8192 d=2 nb=32 hd=64 bf16")
    spec = build_mask(8192, 2, chunk=128)
    Phi, Psi, Vb = _feats(32, 8192, 64, torch.bfloat16, seed=0, q_scale=1 / 8, k_scale=1 / 8,
                          v_scale=1 / 8)
    _check_forward(spec, Phi, Psi, Vb, dt=torch.bfloat16, label="T=8192 d=2")


def test_forward_long_prefill_d3_bf16_T32768():
    """B=1, H=8, head_dim=128, d=3, T=32768, bf16, k scaled 1/sqrt(128); heads 0-1 vs the oracle."""
    _say("forward T=32768 d=3 nb=8 hd=128 bf16")
    T = 32768
    spec = build_mask(T, 3, chunk=128)
    Phi, Psi, Vb = _feats(8, T, 128, torch.bfloat16, seed=0, k_scale=128 ** -0.5)
    out = A.smat_attention(Phi.to(DEV), Psi.to(DEV), Vb.to(DEV), spec)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    _check_forward(spec, Phi[:2], Psi[:2], Vb[:2], dt=torch.bfloat16, label="T=32768 d=3 heads 0-1")
    # heads are independent: a 2-head launch matches the 8-head one (the scan's
    # chunk grouping depends on the batch, so only up to fp32 summation order)
    sub = A.smat_attention(Phi[:2].to(DEV), Psi[:2].to(DEV), Vb[:2].to(DEV), spec)
    assert _rel(sub, out[:2]) < 1e-6
    again = A.smat_attention(Phi.to(DEV), Psi.to(DEV), Vb.to(DEV), spec)
    assert torch.equal(again, out)       # and a repeated launch is bit-identical


def test_forward_long_prefill_d3_bf16_T131072():
    """The benchmark shape (B=1, H=8, head_dim=128, d=3, T=131072, bf16): head 0 vs
    the oracle, and the fused call against the stage-by-stage path."""
    _say("forward T=131072 d=3 nb=8 hd=128 bf16")
    T = 131072
    spec = build_mask(T, 3, chunk=128)
    Phi, Psi, Vb = _feats(8, T, 128, torch.bfloat16, seed=0, k_scale=128 ** -0.5)
    out = A.smat_attention(Phi.to(DEV), Psi.to(DEV), Vb.to(DEV), spec)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    _check_forward(spec, Phi[:1], Psi[:1], Vb[:1], dt=torch.bfloat16, label="T=131072 d=3 head 0")
    staged = A.smat_attention(Phi[:2].to(DEV), Psi[:2].to(DEV), Vb[:2].to(DEV), spec,
                              return_parts=True)
    staged = staged[0] if isinstance(staged, tuple) else staged
    assert _rel(staged, out[:2]) < 1e-5      # one fused call == the stage-by-stage path


def test_forward_long_prefill_d3_bf16_T524288():
    """The largest long-prefill shape (T = 524288, d = 3: q = 67, N0 = 4489, B = 4556,
    the row-group incidence kernel), one head, bf16: against the oracle (the
    reference's torch path on the same bf16 values: 2e-2 on O, 1e-3 on the
    log-normaliser; and the fp64 schedule), the fused call equals the
    stage-by-stage path, and the pooled long-range term equals the direct one
    (each row type summing its landmark outer products without pooling or
    incidence)."""
    _say("forward T=524288 d=3 nb=1 hd=128 bf16")
    T = 524288
    spec = build_mask(T, 3, chunk=128)
    assert (spec.q, spec.N0, spec.B) == (67, 4489, 4556)
    Phi, Psi, Vb = _feats(1, T, 128, torch.bfloat16, seed=5, k_scale=128 ** -0.5)
    Pd, Sd, Wd = Phi.to(DEV), Psi.to(DEV), Vb.to(DEV)
    out = A.smat_attention(Pd, Sd, Wd, spec)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    staged = A.smat_attention(Pd, Sd, Wd, spec, return_parts=True)
    staged = staged[0] if isinstance(staged, tuple) else staged
    assert _rel(staged, out) < 1e-5
    spec_d = A.to_device(spec, DEV, want_direct=True)
    direct = A.smat_attention(Pd, Sd, Wd, spec_d, long_range="direct")
    assert _rel(direct, out) < 1e-5
    del direct, staged
    _check_forward(spec, Phi, Psi, Vb, dt=torch.bfloat16, label="T=524288 d=3 head 0")


@pytest.mark.parametrize("T,heads", [(32768, 2), (131072, 1)])
def test_forward_dense_control_d1_bf16(T, heads):
    """The d = 1 control of the long prefill (B=1, H=8, head_dim=128, bf16, k
    scaled 1/sqrt(128)): M^(1) = L_T, one profile (N0 = 1: its pool is the
    sum of the causal pass's group summaries over [0, n)) and one row type (the query reads one U for all T/2 recent rows).  The
    first heads against the oracle; all heads against the plain causal linear
    attention on the GPU (one unbroken scan, no pool, incidence or query)."""
    _say(f"forward T={T} d=1 nb=8 hd=128 bf16")
    spec = build_mask(T, 1, chunk=128)
    assert (spec.N0, spec.B, spec.n) == (1, 1, T // 2)
    Phi, Psi, Vb = _feats(8, T, 128, torch.bfloat16, seed=0, k_scale=128 ** -0.5)
    Pd, Sd, Wd = Phi.to(DEV), Psi.to(DEV), Vb.to(DEV)
    out = A.smat_attention(Pd, Sd, Wd, spec)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    _check_forward(spec, Phi[:heads], Psi[:heads], Vb[:heads], dt=torch.bfloat16,
                   label=f"T={T} d=1 heads 0-{heads - 1}")
    H = A.segmented_causal_scan(Pd, Sd, Wd, 0, 128)
    plain = H[..., :-1] / H[..., -1:]
    e = _rel(out, plain)
    _say(f"  d=1 vs plain causal: rel {e:.2e}")
    assert e < 1e-4


def test_forward_dense_control_d1_bf16_T524288():
    """d = 1 at T = 524288 (one head, bf16): against the oracle (the reference's
    torch path on the same bf16 values, 2e-2 on O and 1e-3 on the
    log-normaliser, and the fp64 schedule); the fused call equals the staged
    path and equals plain causal linear attention (an unbroken scan)."""
    _say("forward T=524288 d=1 nb=1 hd=128 bf16")
    T = 524288
    spec = build_mask(T, 1, chunk=128)
    Phi, Psi, Vb = _feats(1, T, 128, torch.bfloat16, seed=6, k_scale=128 ** -0.5)
    Pd, Sd, Wd = Phi.to(DEV), Psi.to(DEV), Vb.to(DEV)
    out = A.smat_attention(Pd, Sd, Wd, spec)
    staged = A.smat_attention(Pd, Sd, Wd, spec, return_parts=True)[0]
    H = A.segmented_causal_scan(Pd, Sd, Wd, 0, 128)
    plain = H[..., :-1] / H[..., -1:]
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    e_s, e_p = _rel(staged, out), _rel(out, plain)
    _say(f"  staged {e_s:.2e}  plain causal {e_p:.2e}")
    assert e_s < 1e-5 and e_p < 1e-4
    del staged, H, plain
    _check_forward(spec, Phi, Psi, Vb, dt=torch.bfloat16, label="T=524288 d=1 head 0")


def test_exact_non_influence():
    """A landmark payload outside a recent row's mask leaves that row bit-identical
    (the reference's test_smat.py:292-324, on the GPU path)."""
    _say("non-influence T=2048 d=3 fp32")
    T, d = 2048, 3
    spec = build_mask(T, d, chunk=128)
    Phi, Psi, Vb = _feats(1, T, 32, torch.float32, seed=13)
    base = A.smat_attention(Phi.to(DEV), Psi.to(DEV), Vb.to(DEV), spec).cpu()
    M = __import__("smat_attention_amd.mask", fromlist=["x"]).materialise(spec)
    j = spec.planted_cols[0]
    Vb2 = Vb.clone()
    Vb2[:, j, :-1] += 1e3
    pert = A.smat_attention(Phi.to(DEV), Psi.to(DEV), Vb2.to(DEV), spec).cpu()
    rows_out = [i for i in range(spec.n, T) if M[i, j] == 0]
    rows_in = [i for i in range(spec.n, T) if M[i, j] == 1]
    assert rows_out and rows_in
    assert torch.equal(pert[:, rows_out], base[:, rows_out])
    assert not torch.equal(pert[:, rows_in], base[:, rows_in])


def test_fp64_is_refused():
    _say("fp64 refused")
    spec = build_mask(1024, 2, chunk=128)
    x = torch.rand(1, 1024, 8, device=DEV, dtype=torch.float64)
    with pytest.raises(TypeError):
        A.smat_attention(x, x, torch.rand(1, 1024, 9, device=DEV, dtype=torch.float64), spec)


# ---------------------------------------------------------------------------
# decode
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,d", [(2048, 3), (4096, 2), (1024, 1)])
def test_decode_matches_prefill(dt, T, d):
    _say("decode", dt, T, d)
    spec = build_mask(T, d, chunk=128)
    Phi, Psi, Vb = _feats(3, T, 32, dt, seed=14)
    Pd, Sd, Wd = (x.to(DEV) for x in (Phi, Psi, Vb))
    pre = A.smat_attention(Pd, Sd, Wd, spec).cpu()
    n = spec.n
    dec = A.SmatDecoder(Sd[:, :n], Wd[:, :n], spec)
    steps = min(300, spec.T_R)
    outs = [dec.step(Pd[:, n + i], Sd[:, n + i], Wd[:, n + i]) for i in range(steps)]
    got = torch.stack(outs, 1).cpu()
    ref64 = O.smat_attention(Phi.double(), Psi.double(), Vb.double(), spec)[:, n:n + steps]
    if dt == torch.float32:
        assert _rel(got, ref64) < 1e-5
        assert _rel(got, pre[:, n:n + steps]) < 1e-5
    else:
        assert (got.double() - ref64).abs().max().item() < 2e-2
    assert dec.cache_words() == 3 * (spec.B + 1) * 32 * 33


def test_decode_after_prefill_4096_steps():
    """The cached-decode configuration: B=16, H=8 (nb = 128), head_dim 128, d = 3,
    a 65536-token context, then 4096 steps, bf16 q, k, v ~ N(0, 1) (k scaled
    1/sqrt(128)) from a seeded generator.  The mask is built for the whole
    69632 tokens (q = 37, B = 1406, n = 34816), so every decoded row lies in
    it.  The decoder's U comes from the landmark block, the prefilled recent
    tokens [n, 65536) enter its state in one advance(), then 4096 steps.
    Every decoded row of every sequence is checked against the same row of
    one fused prefill over all 69632 tokens (2e-2 absolute: the prefill rounds
    the in-chunk scores to bf16 as the reference does, the decoder does not),
    and sequences 0-1 against the fp64 oracle's decoder on the same values
    (1e-5 relative: the decoder computes in fp32 from the bf16 values)."""
    nb, hd, T_pre, steps = 128, 128, 65536, 4096
    T = T_pre + steps
    _say(f"decode nb={nb} hd={hd} prefill {T_pre} + {steps} steps bf16")
    spec = build_mask(T, 3, chunk=128)
    assert (spec.q, spec.B, spec.n) == (37, 1406, 34816)
    n = spec.n
    g = torch.Generator(device=DEV).manual_seed(0)
    bf = torch.bfloat16
    Q = torch.randn(nb, T, hd, device=DEV, generator=g).to(bf)
    Kk = (torch.randn(nb, T, hd, device=DEV, generator=g) * hd ** -0.5).to(bf)
    V = torch.randn(nb, T, hd, device=DEV, generator=g).to(bf)
    phi = A.make_phi(hd, hd, device=DEV, dtype=bf, seed=0)
    Phi, Psi, Vb = A.featurise(Q, Kk, V, phi)
    del Q, Kk, V
    pre = A.smat_attention(Phi, Psi, Vb, spec)[:, T_pre:]
    dec = A.SmatDecoder(Psi[:, :n], Vb[:, :n], spec)
    dec.advance(Psi[:, n:T_pre], Vb[:, n:T_pre])
    assert dec.i == T_pre - n
    got = torch.empty(steps, nb, hd, device=DEV)
    for i in range(steps):
        t = T_pre + i
        dec.step(Phi[:, t], Psi[:, t], Vb[:, t], out=got[i])
    torch.cuda.synchronize()
    got = got.transpose(0, 1)
    assert torch.isfinite(got).all()
    e_pre = (got - pre).abs().max().item()
    # sequences 0-1 in fp64: U from the landmark block, the prefilled recent
    # block summed into S, then the oracle's steps
    P2, S2, V2 = (x[:2].double().cpu() for x in (Phi, Psi, Vb))
    ref = O.SmatDecoder(S2[:, :n], V2[:, :n], spec)
    ref.S = S2[:, n:T_pre].transpose(-1, -2) @ V2[:, n:T_pre]
    ref.i = T_pre - n
    want = torch.stack([ref.step(P2[:, T_pre + i], S2[:, T_pre + i], V2[:, T_pre + i])
                        for i in range(steps)], 1)
    e64 = _rel(got[:2], want)
    _say(f"  vs prefill rows {e_pre:.2e} (abs); seqs 0-1 vs fp64 {e64:.2e} (rel)")
    assert e_pre < 2e-2 and e64 < 1e-5


def test_decode_advance_equals_steps():
    """advance() over a block leaves the state and the step counter exactly
    where stepping through the block token by token does (fp32, small)."""
    _say("decode advance vs steps")
    T, d = 4096, 3
    spec = build_mask(T, d, chunk=128)
    Phi, Psi, Vb = _feats(3, T, 32, torch.float32, seed=15)
    Pd, Sd, Wd = (x.to(DEV) for x in (Phi, Psi, Vb))
    n, L = spec.n, 300
    a = A.SmatDecoder(Sd[:, :n], Wd[:, :n], spec)
    b = A.SmatDecoder(Sd[:, :n], Wd[:, :n], spec)
    a.advance(Sd[:, n:n + L], Wd[:, n:n + L])
    for t in range(n, n + L):
        b.step(Pd[:, t], Sd[:, t], Wd[:, t])
    assert a.i == b.i == L
    assert _rel(a.S, b.S) < 1e-6
    oa = torch.stack([a.step(Pd[:, t], Sd[:, t], Wd[:, t]) for t in range(n + L, n + L + 50)], 1)
    ob = torch.stack([b.step(Pd[:, t], Sd[:, t], Wd[:, t]) for t in range(n + L, n + L + 50)], 1)
    assert _rel(oa, ob) < 1e-5


@pytest.mark.parametrize("nb,hd", [(256, 128), (128, 128), (128, 47), (64, 2), (3, 128)])
def test_decode_column_split(nb, hd):
    """The step kernel splits a sequence's value columns over 1, 2 or 4
    workgroups by batch size (256, 128 and 64 sequences here, with odd and
    tiny column counts): every split reproduces the prefill's rows."""
    _say("decode split", nb, hd)
    T = 1024
    spec = build_mask(T, 3, chunk=128)
    Phi, Psi, Vb = _feats(nb, T, hd, torch.float32, seed=15)
    Pd, Sd, Wd = (x.to(DEV) for x in (Phi, Psi, Vb))
    pre = A.smat_attention(Pd, Sd, Wd, spec)
    n = spec.n
    dec = A.SmatDecoder(Sd[:, :n], Wd[:, :n], spec)
    for i in range(24):
        o = dec.step(Pd[:, n + i], Sd[:, n + i], Wd[:, n + i])
        assert _rel(o, pre[:, n + i]) < 1e-5, i


# ---------------------------------------------------------------------------
# the other schedules: endpoint (zeta + Walsh), direct, subtractive
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("N,rp", [(128, 32 * 33), (512, 64 * 65), (4096, 16 * 17), (32768, 8)])
def test_zeta_and_walsh_butterflies(N, rp):
    _say("zeta/walsh", N, rp)
    g = torch.Generator().manual_seed(41)
    F = torch.randn(2, N, rp, generator=g)
    Fd = F.to(DEV)
    Z = A.zeta_transform(Fd.view(2, N, rp, 1))
    W = A.walsh_incidence(Fd.view(2, N, rp, 1))
    Zr = O.zeta_transform(F.double().view(2, N, rp, 1))
    Wr = O.walsh_incidence(F.double().view(2, N, rp, 1))
    assert _rel(Z, Zr) < 1e-5 and _rel(W, Wr) < 1e-5


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,hd", [(256, 32), (300, 32), (1024, 64), (2048, 128)])
def test_forward_endpoint(dt, T, hd):
    """d = floor(log2 T): zeta transform over the landmark block, Walsh incidence."""
    spec = build_mask(T, T.bit_length() - 1, chunk=8)
    assert spec.kind == "endpoint"
    Phi, Psi, Vb = _feats(2, T, hd, dt, seed=42, k_scale=0.5)
    _check_forward(spec, Phi, Psi, Vb, dt=dt, label=f"endpoint T={T} hd={hd}")


@pytest.mark.parametrize("lr", ["direct", "subtractive"])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,d,n_P,hd", [(2048, 3, 0, 32), (2048, 3, 16, 32), (4096, 2, 0, 64),
                                        (8192, 3, 0, 128)])
def test_forward_direct_and_subtractive(lr, dt, T, d, n_P, hd):
    """The comparison schedules against the oracle's own (attention.py:333-362, 458-482)."""
    spec = A.to_device(build_mask(T, d, chunk=128, n_P=n_P), DEV, want_direct=True)
    Phi, Psi, Vb = _feats(2, T, hd, dt, seed=43, k_scale=0.5)
    Pd, Sd, Wd = (x.to(DEV) for x in (Phi, Psi, Vb))
    out = A.smat_attention(Pd, Sd, Wd, spec, long_range=lr)
    torch.cuda.synchronize()
    if dt == torch.float32:
        ref = O.smat_attention(Phi.double(), Psi.double(), Vb.double(), spec, long_range=lr)
        tol = 1e-5 if lr == "direct" else 1e-4      # subtractive cancels in the normaliser
        _say(lr, T, d, n_P, hd, f"fp32 rel {_rel(out, ref):.2e}")
        assert _rel(out, ref) < tol
    else:
        ref = O.smat_attention(Phi, Psi, Vb, spec, long_range=lr)
        e = (out.double().cpu() - ref.double()).abs().max().item()
        _say(lr, T, d, n_P, hd, f"bf16 |O - ref| {e:.2e}")
        assert e < 2e-2
    # the schedules agree with the pooled one
    pooled = A.smat_attention(Pd, Sd, Wd, spec)
    assert (out - pooled).abs().max().item() < (1e-3 if dt == torch.float32 else 3e-2)


def test_direct_head_dim_64_many_items():
    """The direct schedule's unpooled sums (Gram items over landmark column
    lists) at r = 64, p = 65, bf16, 16 sequences -- 2912 items, so the 16-bit
    r = 64 Gram kernel runs -- against the general Gram kernel on the same
    inputs and against the oracle on two sequences."""
    T, d, nb = 4096, 3, 16
    spec = A.to_device(build_mask(T, d, chunk=128), DEV, want_direct=True)
    assert nb * spec.B >= 512
    Phi, Psi, Vb = _feats(nb, T, 64, torch.bfloat16, seed=47, k_scale=0.5)
    Pd, Sd, Wd = (x.to(DEV) for x in (Phi, Psi, Vb))
    _say("direct head_dim 64", T, d, nb)
    out = A.smat_attention(Pd, Sd, Wd, spec, long_range="direct")
    with general_kernel("gram"):
        old = A.smat_attention(Pd, Sd, Wd, spec, long_range="direct")
    torch.cuda.synchronize()
    assert _rel(out, old) < 1e-5
    ref = O.smat_attention(Phi[:2], Psi[:2], Vb[:2], spec, long_range="direct")
    assert (out[:2].double().cpu() - ref.double()).abs().max().item() < 2e-2


def test_decode_endpoint():
    T = 1024
    spec = build_mask(T, T.bit_length() - 1, chunk=8)
    Phi, Psi, Vb = _feats(1, T, 32, torch.float32, seed=44)
    Pd, Sd, Wd = (x.to(DEV) for x in (Phi, Psi, Vb))
    full = A.smat_attention(Pd, Sd, Wd, spec)
    dec = A.SmatDecoder(Sd[:, :spec.n], Wd[:, :spec.n], spec)
    for t in range(spec.n, spec.n + 40):
        o = dec.step(Pd[:, t], Sd[:, t], Wd[:, t])
        assert (o - full[:, t]).abs().max().item() < 1e-4 * max(1.0, full[:, t].abs().max().item())


# ---------------------------------------------------------------------------
# featurise (attention.py:82-106) on HIP
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,dqk,r,dv,kind,gate", [
    (1000, 128, 128, 128, "elu1", True), (777, 64, 64, 64, "elu1", False),
    (130, 32, 48, 7, "relu", True), (64, 40, 16, 33, "elu1", True)])
def test_featurise(dt, T, dqk, r, dv, kind, gate):
    """Phi/Psi/Vb of one HIP launch against the oracle's torch featurise on the
    same inputs.  fp32: relative 1e-5.  16-bit: the product is accumulated in
    another order than torch's, so a rounded product can land one step away
    and elu carries that step on: at most 1e-4 of the outputs may differ by
    more than 2 ulp of the value (2^-7 relative for bf16, 2^-10 for fp16), none
    by more than 4 %.  A wrong rounding order or gate moves far more.  Vb is an
    exact copy."""
    _say("featurise", dt, T, dqk, r, dv, kind, gate)
    g = torch.Generator().manual_seed(31)
    nb = 3
    Q = (torch.randn(nb, T, dqk, generator=g) * 0.5).to(dt)
    K = (torch.randn(nb, T, dqk, generator=g) * 0.5).to(dt)
    V = torch.randn(nb, T, dv, generator=g).to(dt)
    h = (torch.rand(nb, T, generator=g) + 0.5).to(dt) if gate else None
    phi_ref = O.make_phi(dqk, r, kind=kind, dtype=dt, seed=3)
    ref = O.featurise(Q, K, V, phi_ref, h=h)
    phi = A.make_phi(dqk, r, kind=kind, device=DEV, dtype=dt, seed=3)
    got = A.featurise(Q.to(DEV), K.to(DEV), V.to(DEV), phi, h=None if h is None else h.to(DEV))
    for name, a, b in zip(("Phi", "Psi"), got[:2], ref[:2]):
        a = a.cpu().double()
        b = b.double()
        assert a.shape == b.shape
        if dt == torch.float32:
            assert _rel(a, b) < 1e-5, name
        else:
            ulp = 2.0 ** (-7 if dt == torch.bfloat16 else -10)
            rel = (a - b).abs() / b.abs().clamp_min(1e-30)
            assert (rel > ulp).double().mean().item() <= 1e-4, (name, rel.max().item())
            assert rel.max().item() < 0.04, name
    assert torch.equal(got[2].cpu(), ref[2])
    # the map alone, called on a GPU tensor
    assert torch.equal(phi(Q.to(DEV)), got[0])


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_feature_map_every_negative_16_bit_input(dt):
    """The elu + 1 map on every finite non-positive 16-bit input, through the
    featurise launch with W = I (so the product is the input itself), against
    expm1 in fp64 rounded to the dtype, then + 1 rounded (torch's rounding
    steps).  bf16 takes exp2 minus one and must be bit-exact on all 32 641 inputs; fp16 runs libm's expm1f (about 1 ulp of fp32), which may land one
    fp16 step off where the exact value sits within that ulp of a rounding
    boundary: at most 1e-3 of the inputs, by one step."""
    _say("feature map exhaustive", dt)
    itype = torch.int16
    bits = torch.arange(-32768, 32768, dtype=torch.int32).to(itype)
    vals = bits.view(dt).float()
    vals = vals[torch.isfinite(vals) & (vals <= 0)]
    n = vals.numel()
    rows = (n + 127) // 128
    Q = torch.zeros(rows * 128)
    Q[:n] = vals
    Q = Q.reshape(1, rows, 128).to(dt)
    phi = A.FeatureMap(torch.eye(128, device=DEV, dtype=dt), "elu1")
    got = A.featurise(Q.to(DEV), Q.to(DEV), Q.to(DEV), phi)[0].cpu().reshape(-1)[:n]
    v64 = vals.double()
    e = torch.expm1(v64).to(dt)
    want = (e.double() + 1.0).to(dt)
    if dt == torch.bfloat16:
        bad = (got.view(itype) != want.view(itype)).sum().item()
        assert bad == 0, f"{bad} of {n} bf16 inputs differ"
    else:
        step = (got.view(itype).int() - want.view(itype).int()).abs()
        assert step.max().item() <= 1 and (step > 0).double().mean().item() <= 1e-3


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("dqk,r,dv", [(128, 128, 128), (64, 64, 64), (40, 48, 33)])
def test_featurise_of_a_sequence_and_of_a_batch(dqk, r, dv, dt):
    """A call of more row tiles than the GPU has waves (two to a wave) gives, bit for
    bit, the rows of its sequences mapped alone (one to a wave), at a length that
    ends inside a tile and inside a pair; Q, K and V together and Q alone."""
    _say("featurise, one and a batch", dqk, r, dv, dt)
    gen = torch.Generator(device=DEV).manual_seed(93)
    u = lambda *s: torch.randn(*s, device=DEV, generator=gen).to(dt)
    W = (u(r, dqk).float() / dqk ** 0.5).to(dt)
    nb, T = 24, 997
    Q, Kk, V, h = u(nb, T, dqk), u(nb, T, dqk), u(nb, T, dv), u(nb, T)
    many = K.featurise(W, "elu1", Q, Kk, V, h)
    for b in (0, 11, nb - 1):
        one = K.featurise(W, "elu1", Q[b:b + 1], Kk[b:b + 1], V[b:b + 1], h[b:b + 1])
        assert all(torch.equal(x, y[b:b + 1]) for x, y in zip(one, many))
    Q = u(70, T, dqk)
    many = K.featurise(W, "relu", Q)[0]
    for b in (0, 69):
        assert torch.equal(K.featurise(W, "relu", Q[b:b + 1])[0], many[b:b + 1])


def test_featurise_rejects_mixed_dtypes():
    phi = A.make_phi(32, 32, device=DEV, dtype=torch.float32)
    Q = torch.randn(1, 16, 32, device=DEV, dtype=torch.bfloat16)
    with pytest.raises(TypeError):
        A.featurise(Q, Q, Q, phi)



# ---------------------------------------------------------------------------
# the decayed scan (model.py:41-82)
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,n,C,r,p,strength", [
    (1024, 512, 128, 16, 17, 1 / 16), (1000, 500, 64, 32, 33, 1 / 16),
    (4096, 2048, 128, 64, 65, 1 / 16), (512, 256, 128, 128, 129, 2.0), (300, 0, 128, 8, 9, 0.5)])
def test_decayed_scan(dt, T, n, C, r, p, strength):
    """decayed_segmented_scan on HIP against the fp64 oracle on the same values:
    the model's decay logsigmoid(x)/16 and strong decays (weights down to
    e^-250 inside a chunk), a reset inside a chunk, padded tails, head sizes 16
    to 128.  The reference computes in fp32 from upcast inputs, so does this:
    1e-5 relative for every input dtype."""
    _say("decayed scan", dt, T, n, C, r, p, strength)
    g = torch.Generator().manual_seed(T + C + r)
    nb = 3
    Phi = (torch.rand(nb, T, r, generator=g) + 0.1).to(dt)
    Psi = (torch.rand(nb, T, r, generator=g) * 0.2).to(dt)
    Vb = torch.cat([torch.randn(nb, T, p - 1, generator=g), torch.ones(nb, T, 1)], -1).to(dt)
    logA = torch.nn.functional.logsigmoid(torch.randn(nb, T, generator=g)) * strength
    with torch.no_grad():
        got = A.decayed_segmented_scan(Phi.to(DEV), Psi.to(DEV), Vb.to(DEV), logA.to(DEV), n, C)
    ref = O.decayed_segmented_scan(Phi.double(), Psi.double(), Vb.double(), logA.double(), n, C)
    assert torch.isfinite(got).all()
    assert _rel(got.cpu(), ref) < 1e-5


@pytest.mark.parametrize("T,n,C,r,p,strength", [
    (1024, 512, 128, 16, 17, 1 / 16), (1000, 500, 64, 32, 33, 1 / 16),
    (512, 256, 128, 64, 65, 2.0), (300, 0, 128, 8, 9, 0.5)])
def test_decayed_scan_gradients(T, n, C, r, p, strength):
    """The decayed scan's HIP backward: dPhi, dPsi, dVb and dlogA against fp64
    autograd of the oracle on the same fp32 values, within 1e-5 of each
    gradient's largest entry (strong decays, a reset inside a chunk, padded
    tails included)."""
    _say("decayed scan grads", T, n, C, r, p, strength)
    g = torch.Generator().manual_seed(T + C + r + 7)
    nb = 3
    ins = [torch.rand(nb, T, r, generator=g) + 0.1, torch.rand(nb, T, r, generator=g) * 0.2,
           torch.cat([torch.randn(nb, T, p - 1, generator=g), torch.ones(nb, T, 1)], -1),
           torch.nn.functional.logsigmoid(torch.randn(nb, T, generator=g)) * strength]
    R_ = torch.randn(nb, T, p, generator=g)

    def run(dev, dt, f):
        xs = [t.to(dev, dt).requires_grad_(True) for t in ins]
        y = f(*xs)
        (y.float() * R_.to(dev)).sum().backward()
        return y.detach().cpu(), [x.grad.detach().cpu() for x in xs]
    y0, g0 = run("cpu", torch.float64, lambda a, b, c, d: O.decayed_segmented_scan(a, b, c, d, n, C))
    y1, g1 = run(DEV, torch.float32, lambda a, b, c, d: A.decayed_segmented_scan(a, b, c, d, n, C))
    assert _rel(y1, y0) < 1e-5
    for name, a, b in zip(("dPhi", "dPsi", "dVb", "dlogA"), g1, g0):
        assert _rel(a, b) < 1e-5, (name, _rel(a, b))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_forward_identity_incidence_skips_the_gather(dt):
    """At d = 2 the incidence is the identity (row h = [h]): the one-call
    forward queries F directly, bit-identical to running the gather."""
    _say("identity incidence", dt)
    spec = A.to_device(build_mask(4096, 2, chunk=128), DEV)
    assert spec.incidence_identity and spec.n_P == 0
    Phi, Psi, Vb = _feats(2, 4096, 64, dt, seed=50)
    Pd, Sd, Wd = (x.to(DEV) for x in (Phi, Psi, Vb))
    fast = A.smat_attention(Pd, Sd, Wd, spec)
    spec.incidence_identity = False
    try:
        slow = A.smat_attention(Pd, Sd, Wd, spec)
    finally:
        spec.incidence_identity = True
    assert torch.equal(fast, slow)
    # d = 3 keeps the gather, and the C ABI refuses a NULL table for it
    spec3 = A.to_device(build_mask(4096, 3, chunk=128), DEV)
    assert not spec3.incidence_identity
    with pytest.raises(Exception, match="identity incidence"):
        K.forward(Pd, Sd, Wd, None, spec3.uniform_deg, n=spec3.n, n_P=0, N0=spec3.N0,
                  B=spec3.B, chunk=128)


@pytest.mark.parametrize("fused", [False, True])
def test_stage_events_time_the_one_call_forward(fused):
    """smat_set_stage_events: in a one-call forward (plain and fused, T = 8192,
    d = 3, head_dim 128) each stage's last launch binds its event to its end:
    the events come in stage order after one recorded before the call, and the
    output equals a call without events; cleared, later calls leave the
    events as they were."""
    from smat_attention_amd.kernels import _lib
    _say("stage events", fused)
    T = 8192
    spec = build_mask(T, 3, chunk=128)
    gen = torch.Generator().manual_seed(12)
    bf = torch.bfloat16
    Q, K, V = (torch.randn(2, T, 128, generator=gen).to(DEV, bf) for _ in range(3))
    phi = A.FeatureMap(O.phi_weight(128, 128, dtype=bf, seed=0).to(DEV), "elu1")
    Phi, Psi, Vb = A.featurise(Q, K, V, phi)
    run = (lambda: A.smat_attention_fused(Q, K, V, phi, spec)) if fused else \
        (lambda: A.smat_attention(Phi, Psi, Vb, spec))
    plain = run()
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(5)]
    with _lib.stage_events(ev[1:]):
        ev[0].record()
        got = run()
    torch.cuda.synchronize()
    assert torch.equal(got, plain)
    stage = [ev[i].elapsed_time(ev[i + 1]) for i in range(4)]
    _say("  stages (ms)", [round(x, 4) for x in stage])
    assert all(x > 0 for x in stage)
    stamp = ev[0].elapsed_time(ev[4])
    run()
    torch.cuda.synchronize()
    assert ev[0].elapsed_time(ev[4]) == stamp


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("dqk,r,dv", [(64, 64, 64), (128, 128, 128), (40, 96, 33), (64, 48, 8)])
def test_featurise_store_forms_agree(dt, dqk, r, dv):
    """The feature rows stored 16 bytes a lane (16-byte aligned rows, r a multiple of
    32) and value by value (rows at an odd stride) are bitwise the same, at
    lengths beside the 32-row tiles, and no row past the end is written."""
    from smat_attention_amd.kernels.hip_fwd import DTYPE_CODE, call, stream_of
    for T in (1, 15, 16, 31, 32, 33, 65, 200):
        nb = 3
        gen = torch.Generator().manual_seed(T)
        q, k = (torch.randn(nb, T, dqk, generator=gen).to(dt).to(DEV) for _ in range(2))
        v = torch.randn(nb, T, dv, generator=gen).to(dt).to(DEV)
        W = (torch.randn(r, dqk, generator=gen) / dqk ** 0.5).to(dt).to(DEV)
        h = torch.rand(nb, T, generator=gen).to(dt).to(DEV)
        got = []
        for pad, vpad in ((0, (dv + 8) // 8 * 8 - dv), (3, 1)):
            phi, psi = (torch.full((nb, T + 1, r + pad), 7.0, device=DEV, dtype=dt) for _ in range(2))
            vb = torch.full((nb, T + 1, dv + vpad), 7.0, device=DEV, dtype=dt)
            call("smat_featurise", DTYPE_CODE[dt], q.data_ptr(), k.data_ptr(), v.data_ptr(),
                 W.data_ptr(), h.data_ptr(), phi.data_ptr(), psi.data_ptr(), vb.data_ptr(), nb, T, dqk,
                 r, dv, 0, T * dqk, dqk, T * dqk, dqk, T * dv, dv, T, phi.stride(0), phi.stride(1),
                 vb.stride(0), vb.stride(1), stream_of(phi))
            for t, w in ((phi, r), (psi, r), (vb, dv + 1)):
                assert (t[:, T:] == 7).all() and (t[..., w:] == 7).all()
            got.append((phi[:, :T, :r], psi[:, :T, :r], vb[:, :T, :dv + 1]))
        for a, b in zip(*got):
            assert torch.equal(a, b), T
        assert torch.equal(got[0][2][..., :dv], v) and (got[0][2][..., dv] == 1).all()


@pytest.mark.parametrize("dt,hd", [(torch.float32, 64), (torch.float32, 96), (torch.bfloat16, 64),
                                   (torch.float16, 40)])
@pytest.mark.parametrize("T,d,n_P", [(1024, 2, 0), (1000, 3, 0), (2048, 2, 128), (300, 2, 0)])
def test_forward_profile_and_chunk_sums_in_one_launch(dt, hd, T, d, n_P):
    """The one-call forward of a small problem sums its profiles and its chunk groups
    in one launch, a larger one in two: at batch sizes on both sides of that line
    (1024 workgroups at head size 64, 512 above) against the schedule's separate
    launches, whose sums differ only in the order of fp32 additions."""
    _say("pool and prepass", dt, hd, T, d, n_P)
    spec = A.to_device(build_mask(T, d, chunk=128, n_P=n_P), DEV)
    for nb in (1, 3, 7, 12, 24):
        Phi, Psi, Vb = (t.to(DEV) for t in _feats(nb, T, hd, dt, seed=73))
        one = A.smat_attention(Phi, Psi, Vb, spec)
        parts, _ = A.smat_attention(Phi, Psi, Vb, spec, return_parts=True)
        assert _rel(one, parts.double().cpu()) < (2e-5 if dt == torch.float32 else 2.0 ** -7), nb


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("p", [2, 3, 4, 5, 8, 33, 64, 65, 66, 67, 129])
def test_combine_normalise_row_widths(dt, p):
    """The division and its backward at row widths beside the four-value accesses and
    the 64 columns of a pass, rows starting at every alignment, the long-range
    term from row n on: against fp64 (fp32 arithmetic; 2^-8 or 2^-11 more where the
    output is rounded), the floor reached on one row."""
    nb, T, n = 2, 37, 13
    gen = torch.Generator().manual_seed(p)
    H = torch.randn(nb, T, p, generator=gen)
    H[..., -1] = torch.rand(nb, T, generator=gen) + 0.5
    H[0, 3, -1] = -1.0
    Y = torch.rand(nb, T - n, p, generator=gen)
    do = torch.randn(nb, T, p - 1, generator=gen).to(dt)
    Hd, Yd = H.to(DEV).requires_grad_(True), Y.to(DEV).requires_grad_(True)
    out = A.combine_normalise(Hd, Yd, n, out_dtype=dt)
    out.backward(do.to(DEV))
    H64, Y64 = H.double().requires_grad_(True), Y.double().requires_grad_(True)
    N = torch.cat([H64[:, :n], H64[:, n:] + Y64], 1)
    ref = N[..., :-1] / N[..., -1:].clamp_min(1e-6)
    ref.backward(do.double())
    keep = torch.ones(nb, T, dtype=torch.bool)
    keep[0, 3] = False                                # 1e6 times larger: compared by itself
    eps = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -10}[dt]
    got, want = out.detach().cpu().double(), ref.detach()
    assert ((got - want).abs()[keep] <= (1e-5 + eps) * want.abs()[keep] + 1e-5).all()
    for a, b, m in ((Hd.grad, H64.grad, keep), (Yd.grad, Y64.grad, keep[:, n:])):
        assert _rel(a.cpu()[m].to(DEV), b[m]) < 1e-5
    assert _rel(Hd.grad[0, 3, :-1], H64.grad[0, 3, :-1]) < 1e-5 and Hd.grad[0, 3, -1] == 0


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("maxcnt", [0, 64, 100, 400])
def test_query_lists_at_row_block_edges(dt, maxcnt):
    """smat_query_lists at the training shape over lists that end at and beside its
    64-row blocks (empty ones too), with grids sized too small and too large, Y
    rows 65 floats apart: against fp64 within 2e-5 of the largest entry (U enters
    split hi/lo), rows in no list untouched."""
    from smat_attention_amd.kernels.hip_fwd import DTYPE_CODE, call, stream_of
    r, p = 64, 65
    counts = [0, 1, 15, 16, 63, 64, 65, 0, 127, 128, 129, 200]
    L = sum(counts) + 9
    gen = torch.Generator().manual_seed(maxcnt)
    rows = torch.randperm(L, generator=gen)[:sum(counts)]
    X = (torch.rand(L, r, generator=gen) + 0.1).to(dt)
    U = torch.randn(len(counts), r, p, generator=gen)
    Y = torch.full((L, p), 3.0, device=DEV)
    x, u, rw = X.to(DEV), U.to(DEV), rows.int().to(DEV)
    offs = torch.tensor([0] + counts).cumsum(0).to(DEV)
    call("smat_query_lists", DTYPE_CODE[dt], x.data_ptr(), u.data_ptr(), Y.data_ptr(),
         rw.data_ptr(), offs.data_ptr(), len(counts), maxcnt, r, p, r, p, stream_of(Y))
    want = torch.full((L, p), 3.0, dtype=torch.float64)
    kind = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts))
    want[rows] = (X.double()[rows].unsqueeze(1) @ U.double()[kind]).squeeze(1)
    assert _rel(Y, want) < 2e-5
    left = torch.ones(L, dtype=torch.bool)
    left[rows] = False
    assert (Y.cpu()[left] == 3).all()


@pytest.mark.parametrize("T,q,nb", [(5000, 17, 24), (10007, 19, 20), (16384, 23, 14)])
@pytest.mark.parametrize("glob", [False, True])
def test_incidence_line_groups_above_the_cache(T, q, nb, glob):
    """Between q = 17 and 23 F and U of more than 200 MB (600 MB where the forward
    spreads its rows) take one workgroup of 1024 threads a CU, without a global channel:
    the first, a middle and the last sequence are bitwise those of a launch of one
    sequence, which takes the small workgroups (the same sums in the same order)."""
    _say("incidence line groups, large", T, q, nb, glob)
    spec = A.to_device(build_mask(T, 3, chunk=128), DEV)
    assert spec.q == q and nb * (spec.N0 + spec.B) * 128 * 129 * 4 > 768 << 20
    assert (nb // 2) * (spec.N0 + spec.B) * 128 * 129 * 4 < 768 << 20
    g = torch.Generator(device=DEV).manual_seed(q)
    F = torch.randn(nb, spec.N0, 128, 129, device=DEV, generator=g)
    Fg = torch.randn(nb, 128, 129, device=DEV, generator=g) if glob else None
    U = K.incidence_plane(F, spec.plane_code_t, spec.q, F_glob=Fg)
    for i in (0, nb // 2, nb - 1):
        one = K.incidence_plane(F[i:i + 1], spec.plane_code_t, spec.q,
                                F_glob=Fg[i:i + 1] if glob else None)
        assert torch.equal(U[i:i + 1], one), i
