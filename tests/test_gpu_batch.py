"""The batching form (mega_batch_*): uneven cells planned, autotuned and
captured into one hipGraph, checked cell by cell against the single-cell
entry points and the FP64 oracle on cuda:0.

Bars: W bit-identical to mega_zf of the same cell (same group kernel code);
symbols by the parity policy of the FP32 form (x_hat within 1e-4 of the FP64
oracle relative to the symbol's largest |x_hat|, LLRs bit-exact against the
demod of the kernel's own x_hat, hard bits equal away from the boundary);
graph replays bit-identical to the first run."""
import numpy as np
import pytest

import megastation_amd as m
import oracle
from megastation_amd import synth

from gpu_helpers import (SENTINEL, check_symbol, dev_c64, host_c64, host_u16,
                         oracle_llr_from_xhat,
                         llr_buffer, make_slots, oracle_symbol_f64, torch)

pytestmark = pytest.mark.gpu

# U, B, N, sg, Q, layout: every antenna x user size of the uneven-batch
# workload, group sizes 12 and 16, partial last groups, both LLR layouts
CELLS = [
    (8, 64, 624, 12, 4, "standalone"),
    (16, 64, 300, 16, 6, "ldpc"),
    (16, 128, 240, 16, 8, "standalone"),
    (32, 128, 204, 12, 6, "ldpc"),
    (64, 256, 96, 12, 4, "standalone"),
    (8, 64, 100, 16, 8, "standalone"),      # 6.25 groups
    (32, 256, 150, 16, 2, "standalone"),    # 9.4 groups
]


def _make_cells(seed=3, S=2):
    t = torch()
    out = []
    for k, (U, B, N, sg, Q, layout) in enumerate(CELLS):
        sl = make_slots(seed * 100 + k, 1, U, B, N, sg, S, Q, 20.0)[0]
        lay = synth.ldpc_uplink_layout(N, Q) if layout == "ldpc" else synth.standalone_layout(N, Q)
        G = (N + sg - 1) // sg
        out.append(dict(U=U, B=B, N=N, sg=sg, S=S, Q=Q, layout=lay, slot=sl,
                        csi=dev_c64(sl.csi), w=t.zeros(G * B * U, dtype=t.complex64, device="cuda:0"),
                        y=dev_c64(sl.y), llr=llr_buffer(S * U * lay.ue_stride),
                        xhat=t.zeros(S * U * N, dtype=t.complex64, device="cuda:0"),
                        info=t.full((G,), -3, dtype=t.int32, device="cuda:0")))
    return out


def test_batch_matches_single_cell_paths_and_oracle(tmp_path):
    print("case: batch of 7 uneven cells", flush=True)
    t = torch()
    cells = _make_cells()
    cache = str(tmp_path / "tune.txt")
    b = m.Batch(cells, tune_path=cache)
    plan = b.plan()
    print(plan, flush=True)
    b.run()
    t.cuda.synchronize()
    first = [host_u16(c["llr"]).copy() for c in cells]
    for c in cells:
        U, B, N, sg, Q, S, lay = c["U"], c["B"], c["N"], c["sg"], c["Q"], c["S"], c["layout"]
        G = (N + sg - 1) // sg
        assert not c["info"].cpu().numpy().any()
        w1 = t.zeros_like(c["w"])
        m.zf(c["csi"], w1, B, U, G)
        t.cuda.synchronize()
        assert np.array_equal(host_c64(c["w"]), host_c64(w1)), (U, B)
        llr = host_u16(c["llr"]).reshape(S, U, lay.ue_stride)
        xh = host_c64(c["xhat"]).reshape(S, U, N)
        w64, _, _ = oracle.zf(c["slot"].csi, U, B, G, "f64")
        for s in range(S):
            llr64, x64 = oracle_symbol_f64(w64, c["slot"].y[s], U, B, N, sg, Q, lay)
            check_symbol(llr[s], xh[s], llr64, x64, N, sg, Q, lay)
    # replays (graph nodes re-run, counters reset by a kernel) give the same bits
    for _ in range(3):
        for c in cells:
            c["llr"].fill_(SENTINEL)
        b.run()
        t.cuda.synchronize()
        for c, f in zip(cells, first):
            assert np.array_equal(host_u16(c["llr"]), f)
    b.close()
    # a second plan of the same batch takes its tile plans from the cache
    b2 = m.Batch(cells, tune_path=cache)
    assert "(cached)" in b2.plan()
    for c in cells:
        c["llr"].fill_(SENTINEL)
    b2.run()
    t.cuda.synchronize()
    for c, f in zip(cells, first):   # same tile plans -> same arithmetic
        assert np.array_equal(host_u16(c["llr"]), f)
    b2.close()


WIDE_CELLS = [  # every wide tile plan: 1, 2 and 4 user tiles, 64-128 and 160-256 antennas
    (16, 96, 204, 12, 2, "standalone"),
    (20, 64, 100, 16, 4, "ldpc"),
    (33, 96, 77, 8, 6, "standalone"),
    (8, 160, 150, 16, 8, "standalone"),
    (24, 224, 60, 12, 4, "standalone"),
    (50, 160, 41, 12, 8, "standalone"),
]


@pytest.mark.parametrize("cell", [
    (32, 256, 600, 600, 6, "standalone"), (8, 128, 601, 600, 4, "standalone"),
    (40, 64, 700, 300, 2, "ldpc")])
def test_batch_cuts_few_wide_groups_into_many_chunks(cell, tmp_path, monkeypatch):
    """One to three groups of hundreds of column tiles (one of them a single
    subcarrier): the plan cuts them into enough units for the chip, where five
    chunks a group would leave most of it idle."""
    print(f"case: batch few groups {cell}", flush=True)
    t = torch()
    monkeypatch.setitem(globals(), "CELLS", [cell])
    U, B, N, sg, Q, _ = cell
    c, = _make_cells(seed=11, S=7)
    b = m.Batch([c], tune_path=str(tmp_path / "tune.txt"))
    assert "tiles=" in b.plan(), b.plan()
    b.run()
    t.cuda.synchronize()
    b.close()
    w64, _, _ = oracle.zf(c["slot"].csi, U, B, (N + sg - 1) // sg, "f64")
    for s in range(7):
        llr64, x64 = oracle_symbol_f64(w64, c["slot"].y[s], U, B, N, sg, Q, c["layout"])
        check_symbol(host_u16(c["llr"]).reshape(7, U, -1)[s], host_c64(c["xhat"]).reshape(7, U, N)[s],
                     llr64, x64, N, sg, Q, c["layout"])


def test_batch_small_cells_of_one_antenna_count_share_a_class(monkeypatch, tmp_path):
    """Few column tiles: 4 to 64 users of 64 (and of 128) antennas are one equalize
    class, padded to its widest cell's user tiles, with the bits of each cell alone."""
    print("case: batch merged classes", flush=True)
    t = torch()
    monkeypatch.setitem(globals(), "CELLS", [
        (4, 64, 60, 12, 2, "standalone"), (20, 64, 50, 12, 6, "ldpc"), (40, 64, 28, 16, 4, "standalone"),
        (16, 128, 60, 12, 8, "standalone"), (64, 128, 30, 12, 2, "standalone"),
        (17, 128, 24, 8, 4, "standalone")])
    cells = _make_cells(seed=13, S=3)
    outs = []
    for alone in (False, True):
        for c in cells:
            c["llr"].fill_(SENTINEL)
        for k, part in enumerate([[c] for c in cells] if alone else [cells]):
            # the wide form in both (a 64-antenna cell alone may be timed faster
            # with W in one wave's registers, whose sums differ)
            path = tmp_path / f"tune{alone}{k}.txt"
            m.Batch(part, tune_path=str(path)).close()
            keys = [line.split("\t")[0] for line in path.read_text().splitlines()]
            assert len(keys) == (1 if alone else 2)
            mt = {key: max(int(x.split("x")[0]) for x in key.split(";")[1:]) for key in keys}
            path.write_text("".join(
                f"{key}\twide MT={1 if u <= 16 else 2 if u <= 32 else 4} KS=4 chunks=2\n"
                for key, u in mt.items()))
            b = m.Batch(part, tune_path=str(path))
            assert b.plan().count("(cached)") == len(keys)
            b.run()
            t.cuda.synchronize()
            b.close()
        outs.append([(host_u16(c["llr"]).copy(), host_c64(c["xhat"]).copy()) for c in cells])
    for (l0, x0), (l1, x1) in zip(*outs):
        assert np.array_equal(l0, l1) and np.array_equal(x0, x1) and np.abs(x0).max() > 0


def test_batch_wide_plans_of_every_user_tile_count(tmp_path, monkeypatch):
    """As below, each antenna count with cells of one width."""
    monkeypatch.setitem(globals(), "WIDE_CELLS", [
        (16, 96, 204, 12, 2, "standalone"), (8, 160, 150, 16, 8, "standalone"),
        (24, 224, 60, 12, 4, "standalone"), (17, 64, 100, 16, 4, "ldpc"),
        (33, 128, 77, 8, 6, "standalone"), (50, 192, 41, 12, 8, "standalone")])
    test_batch_wide_plans_agree_for_every_chunk_count(tmp_path, monkeypatch)


@pytest.mark.parametrize("cell", [
    (8, 64, 60, 12, 4, "standalone"), (16, 128, 50, 12, 2, "standalone"),
    (32, 256, 30, 12, 6, "standalone"), (50, 96, 31, 16, 8, "standalone")])
def test_batch_infinite_samples(cell, monkeypatch):
    """A received sample of infinite (or overflowing) parts: its column's symbols
    are the four real products' sums, infinities with their signs or NaN where
    they cancel; every other column keeps its bits."""
    print(f"case: batch infinite samples {cell}", flush=True)
    t = torch()
    monkeypatch.setitem(globals(), "CELLS", [cell])
    U, B, N, sg, Q, _ = cell
    c, = _make_cells(seed=21, S=3)
    b = m.Batch([c])
    b.run()
    t.cuda.synchronize()
    clean, llr = host_c64(c["xhat"]).reshape(3, U, N), host_u16(c["llr"]).reshape(3, U, -1).copy()
    y = c["y"].cpu().numpy().reshape(3, B, N).copy()
    y[0, 5, 7] = complex(np.inf, 0.5)
    y[1, B - 1, 0] = complex(0.25, -np.inf)
    y[2, 0, N - 1] = complex(-np.inf, np.inf)
    y[2, B // 2, 20] = complex(3e38, -3e38)  # yi - yr overflows, the products may not
    c["y"].copy_(t.from_numpy(y).reshape(c["y"].shape))
    b.run()
    t.cuda.synchronize()
    b.close()
    got = host_c64(c["xhat"]).reshape(3, U, N)
    got_llr = host_u16(c["llr"]).reshape(3, U, -1)
    w = np.repeat(host_c64(c["w"]).reshape(-1, B, U), sg, axis=0)[:N].astype(np.complex128)
    hit = [(0, 7), (1, 0), (2, N - 1), (2, 20)]
    for s, k in hit:
        x, wk = y[s, :, k].astype(np.complex128), w[k]                       # [B], [B][U]
        with np.errstate(invalid="ignore"):
            re = (wk.real * x.real[:, None] - wk.imag * x.imag[:, None]).sum(0)
            im = (wk.real * x.imag[:, None] + wk.imag * x.real[:, None]).sum(0)
        for g, e in ((got[s, :, k].real, re), (got[s, :, k].imag, im)):
            assert np.array_equal(np.isnan(g), np.isnan(e)), (s, k)
            inf = np.isinf(e)
            assert (g[inf] == e[inf]).all(), (s, k)
            fin = np.isfinite(e) & (np.abs(e) < 3e38)
            assert (np.abs(g[fin] - e[fin]) <= 1e-4 * np.abs(e[fin]).max(initial=0)).all(), (s, k)
    same = np.ones((3, N), bool)
    for s, k in hit:
        same[s, k] = False
        got_llr[s, :, k * Q:(k + 1) * Q] = llr[s, :, k * Q:(k + 1) * Q]
    for s in range(3):
        assert np.array_equal(got[s][:, same[s]], clean[s][:, same[s]])
    assert np.array_equal(got_llr, llr)


@pytest.mark.parametrize("saved", [
    "stream MT=2 waves/CU=12",          # the candidate set before the wide form
    "wide MT=1 KS=4 chunks=4294967295",  # more chunks than 32-bit sums hold
    "wide MT=1 KS=4 chunks=0", "wide MT=2 KS=4 chunks=1", "wide MT=1 KS=8 chunks=1",
    "reg MT=1 KS=8",                    # holds 32 of the 128 antennas
    "reg MT=0 KS=8", "stream MT=0 waves/CU=0"])
def test_batch_measures_saved_plans_that_are_no_candidate(saved, tmp_path, monkeypatch):
    """A line of a tune file that is not one of the class's candidate plans (a
    128-antenna class of 16 users here) is not run: the class is timed again,
    the new choice appended, and the next batch takes that one."""
    print(f"case: batch saved plan {saved!r}", flush=True)
    t = torch()
    monkeypatch.setitem(globals(), "CELLS", [(16, 128, 60, 12, 4, "standalone")])
    cells = _make_cells(seed=9)
    path = tmp_path / "tune.txt"
    path.write_text(f"B=128;16x60/12x2\t{saved}\n")
    b = m.Batch(cells, tune_path=str(path))
    assert "(cached)" not in b.plan()
    b.run()
    t.cuda.synchronize()
    b.close()
    c = cells[0]
    w64, _, _ = oracle.zf(c["slot"].csi, 16, 128, 5, "f64")
    for s in range(c["S"]):
        llr64, x64 = oracle_symbol_f64(w64, c["slot"].y[s], 16, 128, 60, 12, 4, c["layout"])
        check_symbol(host_u16(c["llr"]).reshape(2, 16, -1)[s], host_c64(c["xhat"]).reshape(2, 16, 60)[s],
                     llr64, x64, 60, 12, 4, c["layout"])
    assert len(path.read_text().splitlines()) == 2
    b = m.Batch(cells, tune_path=str(path))
    assert b.plan().count("(cached)") == 1
    b.close()


def test_batch_wide_plans_agree_for_every_chunk_count(tmp_path, monkeypatch):
    """The wide units' results do not depend on how a group's column tiles are
    cut into chunks (1, 2 or 5, forced through the plan file), and match FP64."""
    print("case: batch wide plans", flush=True)
    t = torch()
    monkeypatch.setitem(globals(), "CELLS", WIDE_CELLS)
    cells = _make_cells(seed=5, S=5)
    path = tmp_path / "tune.txt"
    m.Batch(cells, tune_path=str(path)).close()
    saved = [line.split("\t") for line in path.read_text().splitlines()]
    outs = []
    for n in (1, 2, 5):
        with open(path, "w") as f:
            for key, _ in saved:
                B = int(key.split(";")[0][2:])
                U = max(int(c.split("x")[0]) for c in key.split(";")[1:])
                mt = 1 if U <= 16 else 2 if U <= 32 else 4
                f.write(f"{key}\twide MT={mt} KS={4 if B <= 128 else 8} chunks={n}\n")
        for c in cells:
            c["llr"].fill_(SENTINEL)
            c["xhat"].zero_()
        b = m.Batch(cells, tune_path=str(path))
        assert b.plan().count("(cached)") == len(saved)
        b.run()
        t.cuda.synchronize()
        outs.append([(host_u16(c["llr"]).copy(), host_c64(c["xhat"]).copy()) for c in cells])
        b.close()
    for other in outs[1:]:
        for (l0, x0), (l1, x1) in zip(outs[0], other):
            assert np.array_equal(l0, l1) and np.array_equal(x0, x1)
    for c, (llr, xh) in zip(cells, outs[0]):
        U, B, N, sg, Q, S, lay = c["U"], c["B"], c["N"], c["sg"], c["Q"], c["S"], c["layout"]
        w64, _, _ = oracle.zf(c["slot"].csi, U, B, (N + sg - 1) // sg, "f64")
        for s in range(S):
            llr64, x64 = oracle_symbol_f64(w64, c["slot"].y[s], U, B, N, sg, Q, lay)
            check_symbol(llr.reshape(S, U, lay.ue_stride)[s], xh.reshape(S, U, N)[s], llr64, x64,
                         N, sg, Q, lay)


def test_batch_rejects_bad_cells():
    print("case: batch argument checks", flush=True)
    cells = _make_cells()[:2]
    bad = dict(cells[0], Q=5)
    with pytest.raises(m.MegaError) as e:
        m.Batch([cells[1], bad])
    assert e.value.code == m.MEGA_ERR_UNSUPPORTED
    bad = dict(cells[0], U=65)
    with pytest.raises(m.MegaError) as e:
        m.Batch([bad])
    assert e.value.code == m.MEGA_ERR_UNSUPPORTED


def _gpu_cell(cfg, seed):
    """Inputs of one cell generated on the GPU: A = H^H [G][B][U] (i.i.d.
    CN(0,1)), y = H x + n [S][B][N] at the cell's SNR, x from the QAM table."""
    t = torch()
    U, B, N, sg, S, Q = (cfg[k] for k in ("U", "B", "N", "sg", "S", "Q"))
    G = (N + sg - 1) // sg
    gen = t.Generator(device="cuda:0")
    gen.manual_seed(seed)
    H = t.randn((G, B, U), dtype=t.complex64, device="cuda:0", generator=gen)
    table = t.from_numpy(synth.qam_table(Q)).to("cuda:0")
    x = table[t.randint(0, 1 << Q, (S, U, G * sg), device="cuda:0", generator=gen)]
    X = x.reshape(S, U, G, sg).permute(2, 1, 0, 3).reshape(G, U, S * sg).contiguous()
    Hr, Hi, Xr, Xi = (v.contiguous() for v in (H.real, H.imag, X.real, X.imag))
    Y = t.complex(t.bmm(Hr, Xr) - t.bmm(Hi, Xi), t.bmm(Hr, Xi) + t.bmm(Hi, Xr))
    Y = Y + (10 ** (-cfg["snr"] / 20)) * t.randn(Y.shape, dtype=t.complex64, device="cuda:0",
                                                  generator=gen)
    y = Y.reshape(G, B, S, sg).permute(2, 1, 0, 3).reshape(S, B, G * sg)[..., :N].contiguous()
    csi = t.conj(H).resolve_conj().contiguous()
    return csi, y, x[..., :N].contiguous()


def test_batch_40_uneven_cells_full_size():
    """The uneven 40-cell workload at its full sizes (13 symbols, N up to
    3276, 256 x 64 cells, QAM 16/64/256, partial last groups): every cell's W
    bit-identical to mega_zf; every symbol's LLRs bit-identical to the
    oracle's demod and placement of the kernel's own x_hat; symbols 0 and 12
    of every cell within the FP64 bar (x_hat within 1e-4 of FP64 zero-forcing
    relative to the symbol's largest |x_hat|, EVM within 0.1 dB)."""
    t = torch()
    cfgs = synth.uneven_cells(40, 7)
    print(f"case: batch of 40 uneven cells, full size", flush=True)
    cells = []
    for k, cfg in enumerate(cfgs):
        U, B, N, sg, S, Q = (cfg[x] for x in ("U", "B", "N", "sg", "S", "Q"))
        G = (N + sg - 1) // sg
        csi, y, x = _gpu_cell(cfg, 1000 + k)
        lay = synth.standalone_layout(N, Q)
        cells.append(dict(U=U, B=B, N=N, sg=sg, S=S, Q=Q, layout=lay, csi=csi, y=y, x=x,
                          w=t.zeros(G * B * U, dtype=t.complex64, device="cuda:0"),
                          llr=llr_buffer(S * U * lay.ue_stride),
                          xhat=t.zeros(S * U * N, dtype=t.complex64, device="cuda:0"),
                          info=t.full((G,), -3, dtype=t.int32, device="cuda:0")))
    b = m.Batch(cells)
    print(b.plan(), flush=True)
    b.run()
    t.cuda.synchronize()
    for k, c in enumerate(cells):
        U, B, N, sg, Q, S, lay = c["U"], c["B"], c["N"], c["sg"], c["Q"], c["S"], c["layout"]
        G = (N + sg - 1) // sg
        print(f"  cell {k}: {B}x{U} N={N} sg={sg} Q={Q}", flush=True)
        assert not c["info"].cpu().numpy().any()
        w1 = t.zeros_like(c["w"])
        m.zf(c["csi"], w1, B, U, G)
        t.cuda.synchronize()
        assert np.array_equal(host_c64(c["w"]), host_c64(w1)), k
        llr = host_u16(c["llr"]).reshape(S, U, lay.ue_stride)
        xh = host_c64(c["xhat"]).reshape(S, U, N)
        for s in range(S):
            assert np.array_equal(llr[s], oracle_llr_from_xhat(xh[s], N, sg, Q, lay)), (k, s)
        # FP64 zero-forcing (numpy complex128) of symbols 0 and S-1
        A = host_c64(c["csi"]).astype(np.complex128).reshape(G, B, U).transpose(0, 2, 1)
        W64 = np.linalg.solve(A @ A.conj().transpose(0, 2, 1), A)       # [G][U][B]
        yh = host_c64(c["y"]).reshape(S, B, N)
        xt = host_c64(c["x"]).reshape(S, U, N)
        for s in (0, S - 1):
            yp = np.zeros((B, G * sg), np.complex128)
            yp[:, :N] = yh[s]
            x64 = (W64 @ yp.reshape(B, G, sg).transpose(1, 0, 2)).transpose(1, 0, 2)
            x64 = x64.reshape(U, G * sg)[:, :N]
            err = np.abs(xh[s] - x64).max() / np.abs(x64).max()
            assert err < 1e-4, (k, s, err)
            e_gpu, e_64 = synth.evm_db(xh[s], xt[s]), synth.evm_db(x64, xt[s])
            assert abs(e_gpu - e_64) < 0.1, (k, s, e_gpu, e_64)
    b.close()
