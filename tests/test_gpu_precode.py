"""Downlink precode on cuda:0 (mega_precode / mega_precode_syms) against the
oracle (orc_precode, pinned to the reference's test/sgemv/precoded.data) and
the reference fixture itself. FP32 products: the bar is the reference test's
1e-5 (relative to the output scale for the large shapes). Output buffers are
prefilled with a sentinel, so the entries the reference leaves untouched
(guard columns, a partial last group) are checked too."""
import numpy as np
import pytest

import megastation_amd as m
import oracle

from gpu_helpers import dev_c64, host_c64, torch

pytestmark = pytest.mark.gpu

SENT = np.complex64(7 - 3j)


def test_precode_reference_fixture(golden):
    print("case: precode reference fixture 8x4, 16 subcarriers, row 32", flush=True)
    t = torch()
    prec = dev_c64(golden["precode_prec"])
    ue = dev_c64(golden["precode_uevec_ku"].reshape(16, 4).T.copy().reshape(-1))
    out = t.zeros(8 * 32, dtype=t.complex64, device="cuda:0")
    rc = m.lib().mega_precode(8, 4, 16, m._ptr(prec), m._ptr(ue), m._ptr(out), 32, 16, 8,
                              m._stream(None))
    assert rc == 0, m.last_error()
    t.cuda.synchronize()
    got = host_c64(out).reshape(8, 32)
    assert np.abs(got - golden["precode_out"].reshape(8, 32)).max() < 1e-5


@pytest.mark.parametrize("B,U,N,sg,row,start,S", [
    (64, 16, 1200, 16, 2048, 424, 1),    # the reference's PrecodeLarge shape
    (256, 32, 3276, 12, 4096, 410, 3),   # 256x32 cell, 273 groups, three symbols
    (24, 5, 100, 12, 128, 17, 2),        # partial last group left untouched
    (130, 64, 200, 40, 256, 0, 1),       # sg > 32 (column chunks), 64 users
    (8, 3, 7, 8, 16, 3, 1),              # no full group: nothing written
])
def test_precode_matches_oracle(B, U, N, sg, row, start, S):
    print(f"case: precode B={B} U={U} N={N} sg={sg} row={row} start={start} S={S}", flush=True)
    t = torch()
    rng = np.random.default_rng(B * 7 + U + N)
    G = max(1, N // sg)
    P = (rng.standard_normal((G, U, B)) + 1j * rng.standard_normal((G, U, B))).astype(np.complex64)
    ue_pad, out_pad = U * N + 5, B * row + 3  # padded symbol strides
    ue = np.zeros((S, ue_pad), np.complex64)
    ue[:, :U * N] = (rng.standard_normal((S, U * N)) + 1j * rng.standard_normal((S, U * N)))
    out = t.from_numpy(np.full(S * out_pad, SENT, np.complex64)).to("cuda:0")
    m.precode(dev_c64(P.reshape(-1)), dev_c64(ue.reshape(-1)), out, num_bs=B, num_ue=U,
              num_sc=N, sc_group=sg, bs_stride=row, bs_start=start, num_syms=S,
              ue_sym_stride=ue_pad, bs_sym_stride=out_pad)
    t.cuda.synchronize()
    got = host_c64(out).reshape(S, out_pad)
    for s in range(S):
        fill = np.full((B, row), SENT, np.complex64)
        exp = oracle.precode(P, ue[s, :U * N].reshape(U, N), B, U, N, sg, row, start, out=fill)
        g = got[s, :B * row].reshape(B, row)
        untouched = exp == SENT
        assert np.array_equal(g[untouched], exp[untouched])
        scale = max(1.0, float(np.abs(exp[~untouched]).max(initial=0.0)))
        np.testing.assert_allclose(g, exp, rtol=1e-5, atol=1e-5 * scale)
        assert (got[s, B * row:] == SENT).all()  # stride padding untouched
    if N < sg:
        assert (got == SENT).all()



@pytest.mark.parametrize("B,U,N,sg,row,start,S", [
    (97, 40, 500, 8, 512, 6, 14),    # 33-64 users, 434 tiles over two antenna blocks' ranges
    (300, 20, 333, 7, 512, 300, 3),  # the shift wraps round the row; three antenna blocks
    (200, 32, 1637, 12, 2048, 205, 14),  # ranges that cross groups at every place of a tile
    (1, 1, 40, 3, 64, 1, 1),
])
def test_precode_ranges_match_fp64(B, U, N, sg, row, start, S):
    """The register kernel's ranges, antenna blocks and user steps: FP32 sums
    of U products, so within U * 2^-23 of the sum of magnitudes; untouched
    columns stay."""
    print(f"case: precode ranges B={B} U={U} N={N} sg={sg} S={S}", flush=True)
    t = torch()
    rng = np.random.default_rng(B + U + N)
    G, full = -(-N // sg), N // sg
    P = (rng.standard_normal((G, U, B)) + 1j * rng.standard_normal((G, U, B))).astype(np.complex64)
    ue = (rng.standard_normal((S, U, N)) + 1j * rng.standard_normal((S, U, N))).astype(np.complex64)
    out = t.from_numpy(np.full((S, B, row), SENT, np.complex64)).to("cuda:0")
    m.precode(dev_c64(P.reshape(-1)), dev_c64(ue.reshape(-1)), out, num_bs=B, num_ue=U, num_sc=N,
              sc_group=sg, bs_stride=row, bs_start=start, num_syms=S)
    got = host_c64(out).reshape(S, B, row)
    exp = np.full((S, B, row), SENT, np.complex128)
    mag = np.zeros((S, B, row))
    for g in range(full):
        k = np.arange(g * sg, (g + 1) * sg)
        col = (k + start + row // 2) % row
        exp[:, :, col] = np.einsum("ub,suk->sbk", P[g].astype(np.complex128), ue[:, :, k])
        mag[:, :, col] = np.einsum("ub,suk->sbk", np.abs(P[g]), np.abs(ue[:, :, k]))
    untouched = mag == 0
    assert np.array_equal(got[untouched], exp[untouched].astype(np.complex64))
    assert (np.abs(got - exp) <= 4 * U * 2.0 ** -23 * mag + 1e-30).all()


@pytest.mark.parametrize("B,U,N,sg,S", [
    (256, 3, 3276, 12, 13), (300, 7, 1650, 12, 13), (256, 13, 3276, 12, 13),  # tiles dealt round
    (300, 21, 3276, 12, 13),                                                  # a group a wave
    (160, 30, 3276, 12, 13), (200, 9, 3277, 12, 13), (96, 45, 3276, 12, 5),   # ranges of groups
    (128, 10, 3280, 16, 14), (70, 61, 4000, 9, 14),                           # equal ranges
])
def test_precode_divisions_of_the_work_match_fp64(B, U, N, sg, S):
    """Every way to divide a full slot's tiles and antenna blocks among waves,
    with the bound of the test above."""
    print(f"case: precode division B={B} U={U} N={N} sg={sg} S={S}", flush=True)
    t = torch()
    gen = t.Generator(device="cuda").manual_seed(B + U)
    G = N // sg
    P = t.randn(-(-N // sg), U, B, dtype=t.complex64, device="cuda", generator=gen)
    ue = t.randn(S, U, N, dtype=t.complex64, device="cuda", generator=gen)
    out = t.full((S, B, N + 3), complex(SENT), dtype=t.complex64, device="cuda")
    half = (N + 3) // 2
    m.precode(P, ue, out, num_bs=B, num_ue=U, num_sc=N, sc_group=sg, bs_stride=N + 3,
              bs_start=N + 3 - half, num_syms=S)  # the columns as they are
    A = P[:G].transpose(1, 2).to(t.complex128).contiguous()                  # [G][B][U]
    X = ue[:, :, :G * sg].reshape(S, U, G, sg).permute(2, 1, 0, 3).reshape(G, U, S * sg)
    X = X.to(t.complex128).contiguous()
    unfold = lambda y: y.reshape(G, B, S, sg).permute(2, 1, 0, 3).reshape(S, B, G * sg)
    err = (out[:, :, :G * sg] - unfold(A @ X)).abs()
    assert bool((err <= 4 * U * 2.0 ** -23 * unfold(A.abs() @ X.abs())).all())
    assert bool((out[:, :, G * sg:] == complex(SENT)).all())


@pytest.mark.parametrize("U,B", [(2, 40), (6, 200), (17, 64), (18, 130), (34, 70)])
def test_precode_infinities_of_the_last_user(U, B):
    """Users are padded to whole steps: an infinite entry or symbol of the last
    one gives the products' infinities, not the NaN of a padded zero times it."""
    print(f"case: precode infinities U={U} B={B}", flush=True)
    rng = np.random.default_rng(U)
    N, sg = 48, 12
    t = torch()
    draw = lambda *s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)
    P, ue = draw(N // sg, U, B), draw(1, U, N)
    P[1, U - 1, ::3] = np.inf + 1j
    ue[0, U - 1, 30::5] = complex(2, -np.inf)
    out = t.zeros(B, N, dtype=t.complex64, device="cuda:0")
    m.precode(dev_c64(P.reshape(-1)), dev_c64(ue.reshape(-1)), out, num_bs=B, num_ue=U, num_sc=N,
              sc_group=sg, bs_stride=N, bs_start=N // 2, num_syms=1)
    got = host_c64(out).reshape(B, N)
    Pk = np.repeat(P, sg, axis=0).astype(np.complex128)       # [N][U][B]
    x = ue[0].T[:, :, None].astype(np.complex128)             # [N][U][1]
    re = (Pk.real * x.real - Pk.imag * x.imag).sum(1).T       # real products, as in the kernel
    im = (Pk.real * x.imag + Pk.imag * x.real).sum(1).T
    assert np.isinf(re).any() and np.isinf(im).any()
    for g, e in ((got.real, re), (got.imag, im)):
        fin = np.isfinite(e)
        assert np.isinf(e[~fin]).all() and (g[~fin] == e[~fin]).all()
        assert np.isfinite(g[fin]).all()


def test_precode_group_beyond_32_bit_byte_offsets():
    """One group's precoder of 4 GiB and a little: antennas past 2^29 read their
    own entries (times 2: exact)."""
    B = 2**29 + 40
    print(f"case: precode B={B} U=1", flush=True)
    t = torch()
    P = t.zeros(B, 2, device="cuda:0")
    P[:, 0] = t.arange(B, device="cuda:0", dtype=t.float32)
    P[:, 1] = 1.0
    ue = t.full((1,), 2.0 + 0j, dtype=t.complex64, device="cuda:0")
    out = t.full((B, 2), -1.0, device="cuda:0")
    m.precode(P, ue, out, num_bs=B, num_ue=1, num_sc=1, sc_group=1, bs_stride=1, bs_start=0,
              num_syms=1)
    P *= 2
    for lo in range(0, B, 2**26):
        assert t.equal(out[lo:lo + 2**26], P[lo:lo + 2**26]), lo


@pytest.mark.parametrize("U,B,G", [
    (8, 8, 5), (5, 13, 7), (2, 1, 300000), (16, 16, 9), (1, 250, 3),  # a wave a group
    (1, 257, 3), (3, 171, 2), (16, 64, 70000),                        # one LDS tile
    (4, 5000, 2), (16, 1100, 2), (3, 11011, 2), (130, 128, 2)])       # several
def test_precoder_normalisation_of_small_and_tall_groups(U, B, G):
    """As below, against torch in 64 bits; and groups of zeros, of an infinity and
    with a NaN (which the maximum passes over) give what the expression gives."""
    print(f"case: precoder normalisation U={U} B={B} G={G}", flush=True)
    t = torch()
    W = t.randn(G, B, U, dtype=t.complex64, device="cuda",
                generator=t.Generator(device="cuda").manual_seed(U + B))
    W[1] = 0
    W[0, B // 2, U // 2] = complex(np.inf, 1)
    if G > 2 and U * B > 2:
        W[2, B - 1, U - 1] = complex(np.nan, 2)
    P = t.zeros(G, U, B, dtype=t.complex64, device="cuda")
    m.Beamform.beamform_downlink(W, P, U, B, G)
    w = W.to(t.complex128)
    mag = t.nan_to_num(w.abs(), nan=0.0, posinf=np.inf).amax((1, 2), keepdim=True)
    for got, part in ((P.real, w.real), (P.imag, w.imag)):
        e = (part / mag).transpose(1, 2)
        assert bool(((got - e).abs()[3:] < 4 * 2.0 ** -23).all())
        for g in range(min(3, G)):
            fin = t.isfinite(e[g]) & t.isfinite(w[g].real.T) & t.isfinite(w[g].imag.T)
            assert bool(((got[g] - e[g]).abs()[fin] < 4 * 2.0 ** -23).all())
            assert not bool(t.isfinite(got[g][~fin]).any())


@pytest.mark.parametrize("U,B,G", [(1, 1, 3), (32, 256, 5), (64, 256, 2), (128, 300, 2), (100, 1, 4),
                                   (17000, 2, 1)])
def test_precoder_normalisation_shapes(U, B, G):
    """One LDS tile, several tiles and none: P = W^T / max|W| within the two
    roundings of 1 / max and the product."""
    print(f"case: precoder normalisation U={U} B={B} G={G}", flush=True)
    t = torch()
    rng = np.random.default_rng(U + B)
    W = (rng.standard_normal((G, B, U)) + 1j * rng.standard_normal((G, B, U))).astype(np.complex64)
    P = t.zeros(G, U, B, dtype=t.complex64, device="cuda:0")
    m.Beamform.beamform_downlink(dev_c64(W.reshape(-1)), P, U, B, G)
    got = host_c64(P).reshape(G, U, B)
    exp = (W / np.abs(W.astype(np.complex128)).max((1, 2), keepdims=True)).swapaxes(1, 2)
    assert np.abs(got - exp).max() < 4 * 2.0 ** -23
