"""Timed cases of the framework's public entry points: the uplink detection
path (ZF weights, equalize + demod) in its plain, pipelined, batched and
learned forms, the uplink from received samples, the downlink precode and
IFFT, the LDPC decoder, and a training step of the warm-start network.

listed() gives the fixed cases, draw(rng) one more of the same ranges;
prepare(case, seed) makes inputs on the GPU from the seed alone, run(state)
is one pass, work(case) what a pass cannot do without, exact(case, seed) the
outputs in 64 bits from plain torch / numpy.
"""
import math
import os

import numpy as np
import torch

import megastation_amd as m
from megastation_amd import learned, pipeline, synth

DEV = "cuda:0"
CKPT = os.path.join(os.path.dirname(os.path.abspath(learned.__file__)), "data",
                    "warmstart_128x32.npz")


def listed():
    return [
        # One slot of the reference's own 64 x 16 cell (16 users, 1200
        # subcarriers, 16-QAM, the LDPC layout its pipeline hands over): the
        # smallest call, where latency and launches count.
        dict(name="slot_64x16", kind="slots", U=16, B=64, N=1200, sg=16, S=13, Q=4, slots=1,
             form="fp32", channel="iid", snr=20.0, layout="ldpc"),
        # The same cell with 200 slots a call, as a base station with many
        # cells or an offline run batches it: bound by memory.
        dict(name="slots_64x16x200", kind="slots", U=16, B=64, N=1200, sg=16, S=13, Q=4,
             slots=200, form="fp32", channel="iid", snr=20.0, layout="standalone"),
        # One slot of the 256 x 32 massive-MIMO cell through the drop-in
        # entry points: ZF, then equalize + demod.
        dict(name="slot_256x32", kind="slots", U=32, B=256, N=3276, sg=12, S=13, Q=6, slots=1,
             form="fp32", channel="kronecker", snr=25.0, layout="standalone"),
        # Eight consecutive slots of that cell in the mixed form, bound to a
        # pipeline graph: a serving loop's steady state.
        dict(name="graph_256x32_mixed", kind="graph", U=32, B=256, N=3276, sg=12, S=13, Q=6,
             pushes=8, form="mixed", channel="kronecker", snr=25.0, layout="standalone"),
        # A cell whose sizes are no powers of two: 48 users on 200 antennas,
        # a partial last group, 256-QAM.
        dict(name="slot_200x48_ragged", kind="slots", U=48, B=200, N=1637, sg=12, S=13, Q=8,
             slots=1, form="fp32", channel="iid", snr=28.0, layout="standalone"),
        # Forty cells of uneven shapes in one launch of a batch handle.
        dict(name="batch_40cells", kind="batch", cells=40, pick=7),
        # A whole uplink slot of the 256 x 32 cell from received int16
        # samples: pilot FFT to CSI, ZF, data FFT, equalize + demod.
        dict(name="uplink_256x32", kind="uplink", U=32, B=256, ca=4096, N=3276, sg=12, S=13,
             Q=6, bits=16, snr=25.0),
        # The downlink of that cell: the precoder from W, and 13 symbols
        # precoded into 4096-point rows.
        dict(name="precode_256x32", kind="precode", U=32, B=256, ca=4096, N=3276, sg=12, S=13),
        # The downlink's last stage: precoded rows to int16 samples.
        dict(name="ifft_256x4096", kind="ifft", B=256, ca=4096, N=3276, S=13, bits=16),
        # The code blocks of a 256 x 32 slot (32 users x 13 symbols), BG1 at
        # rate 1/3, binary16 LLRs in the equalizer's padded rows.
        dict(name="ldpc_256x32", kind="ldpc", bg=1, zc=288, mb=46, iters=8, cb=416, bits=16),
        # One slot of the learned form on a time-varying channel: warm-start
        # network, Newton-Schulz, fallback, then equalize + demod.
        dict(name="learned_128x32", kind="learned", U=32, B=128, N=3276, sg=12, S=13, Q=6,
             snr=25.0),
        # One training step of that network on four slot pairs: forward,
        # backward, Adam.
        dict(name="train_32users", kind="train", U=32, B=128, G=273, pairs=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["slots", "slots", "slots", "graph", "batch", "uplink", "precode", "ifft",
                       "ldpc", "learned", "train"])
    U = _log(rng, 4, 64)
    B = min(256, _log(rng, max(2 * U, 16), 256))
    if U > 32:
        B = rng.randint(max(128, 2 * U), 256)
    sg, S, Q = rng.choice([8, 12, 16]), rng.randint(7, 14), rng.choice([2, 4, 6, 8])
    N = _log(rng, 300, 3276)
    if kind == "slots":
        most = max(1, min(200, int(150e6 // (B * N * S))))
        return dict(kind=kind, U=U, B=B, N=N, sg=sg, S=S, Q=Q, slots=_log(rng, 1, most),
                    form=rng.choice(["fp32", "fp32", "mixed"]),
                    channel=rng.choice(["iid", "kronecker"]), snr=float(rng.randint(10, 30)),
                    layout=rng.choice(["standalone", "ldpc"]))
    if kind == "graph":
        return dict(kind=kind, U=U, B=B, N=N, sg=sg, S=S, Q=Q, pushes=rng.randint(2, 8),
                    form=rng.choice(["fp32", "mixed"]), channel="iid",
                    snr=float(rng.randint(10, 30)), layout="standalone")
    if kind == "batch":
        return dict(kind=kind, cells=_log(rng, 3, 40), pick=rng.randint(100, 10 ** 6))
    if kind in ("uplink", "ifft", "precode"):
        ca = rng.choice([512, 1024, 2048, 4096])
        N = rng.randint(ca // 2, ca * 4 // 5)
        if kind == "uplink":
            # whole groups only: a user without a pilot in a partial last
            # group would have no channel estimate there
            return dict(kind=kind, U=U, B=B, ca=ca, N=N // sg * sg, sg=sg, S=S, Q=Q,
                        bits=rng.choice([16, 16, 8]), snr=float(rng.randint(10, 30)))
        if kind == "ifft":
            return dict(kind=kind, B=_log(rng, 8, 256), ca=ca, N=N, S=S,
                        bits=rng.choice([16, 16, 8]))
        return dict(kind=kind, U=U, B=B, ca=ca, N=N, sg=sg, S=S)
    if kind == "ldpc":
        bg = rng.choice([1, 1, 2])
        zc = rng.choice([z for z in synth.LDPC_ZC if z >= 24])
        return dict(kind=kind, bg=bg, zc=zc, mb=rng.randint(8, 46 if bg == 1 else 42),
                    iters=rng.randint(4, 12), cb=_log(rng, 8, 600), bits=rng.choice([16, 16, 32]))
    if kind == "learned":
        return dict(kind=kind, U=32, B=rng.randint(96, 192), N=rng.randint(600, 3276), sg=12,
                    S=S, Q=rng.choice([4, 6, 8]), snr=float(rng.randint(15, 30)))
    return dict(kind="train", U=rng.choice([8, 16, 24, 32]), B=rng.choice([64, 128]),
                G=rng.randint(60, 273), pairs=rng.randint(1, 4))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _cn(gen, *shape):
    """CN(0, 1) complex64."""
    return torch.randn(shape, dtype=torch.complex64, device=DEV, generator=gen)


def _groups(N, sg):
    return (N + sg - 1) // sg


def _mul(a, b):
    """Batched complex product on contiguous real parts."""
    ar, ai, br, bi = (t.contiguous() for t in (a.real, a.imag, b.real, b.imag))
    return torch.complex(torch.bmm(ar, br) - torch.bmm(ai, bi),
                         torch.bmm(ar, bi) + torch.bmm(ai, br))


def _channel(gen, n, B, U, kind):
    """H [n][B][U]: CN(0, 1), or with exponential correlation 0.5 / 0.3
    between antennas / users."""
    H = _cn(gen, n, B, U)
    if kind == "kronecker":
        def root(k, rho):
            w, v = np.linalg.eigh(synth.exp_corr(k, rho))
            r = ((v * np.sqrt(np.maximum(w, 0))) @ v.T).astype(np.float32)
            return torch.from_numpy(r).to(DEV)
        rx, tx = root(B, 0.5), root(U, 0.3)
        re = torch.matmul(torch.matmul(rx, H.real.contiguous()), tx)
        im = torch.matmul(torch.matmul(rx, H.imag.contiguous()), tx)
        H = torch.complex(re, im)
    return H


def _symbols(gen, Q, *shape):
    table = torch.from_numpy(synth.qam_table(Q)).to(DEV)
    return table[torch.randint(0, 1 << Q, shape, device=DEV, generator=gen)]


def _received(gen, H, slots, N, sg, S, Q, snr):
    """y [slots][S][B][N] = H x + noise for H [slots*G][B][U]."""
    n, B, U = H.shape
    G = n // slots
    x = _symbols(gen, Q, n, U, S * sg)
    y = _mul(H, x)
    y += 10.0 ** (-snr / 20.0) * _cn(gen, *y.shape)
    y = y.reshape(slots, G, B, S, sg).permute(0, 3, 2, 1, 4)
    return y.reshape(slots, S, B, G * sg)[..., :N].contiguous()


def _csi(H):
    return torch.conj(H).resolve_conj().contiguous()


def _layout(c):
    if c.get("layout") == "ldpc":
        return synth.ldpc_uplink_layout(c["N"], c["Q"])
    return synth.standalone_layout(c["N"], c["Q"])


def _place(c, lay):
    return dict(ue_stride=lay.ue_stride, cb_size=lay.cb_size, cb_stride=lay.cb_stride,
                zeros=lay.zeros, valid_bits=lay.valid_bits)


def _form(c):
    return m.FORM_MIXED if c["form"] == "mixed" else m.FORM_FP32


def _slot_inputs(c, seed, slots):
    """(csi [slots*G][B][U], y [slots][S][B][N])."""
    gen = _gen(seed)
    G = _groups(c["N"], c["sg"])
    H = _channel(gen, slots * G, c["B"], c["U"], c["channel"])
    return _csi(H), _received(gen, H, slots, c["N"], c["sg"], c["S"], c["Q"], c["snr"])


def _slots(c, seed):
    U, B, N, sg, S, Q, n = (c[k] for k in ("U", "B", "N", "sg", "S", "Q", "slots"))
    G, lay, form = _groups(N, sg), _layout(c), _form(c)
    csi, y = _slot_inputs(c, seed, n)
    llr = torch.zeros(n * S * U * lay.ue_stride, dtype=torch.int16, device=DEV)
    if form == m.FORM_MIXED:
        Bp = (B + 15) // 16 * 16
        w, wstride = torch.zeros(n * G * U * Bp, dtype=torch.int64, device=DEV), G * U * Bp
    else:
        w, wstride = torch.zeros(n * G * B * U, dtype=torch.complex64, device=DEV), G * B * U
    eq = dict(num_ue=U, num_bs=B, num_sc=N, sc_group=sg, num_syms=S, num_slots=n, mod_order=Q,
              csi_slot_stride=wstride, y_sym_stride=B * N, y_slot_stride=S * B * N,
              llr_sym_stride=U * lay.ue_stride, llr_slot_stride=S * U * lay.ue_stride,
              form=form, **_place(c, lay))
    return dict(kind="slots", csi=csi, y=y, w=w, llr=llr, B=B, U=U, n=n * G, eq=eq, form=form)


def _run_slots(s):
    if s["form"] == m.FORM_MIXED:
        m.zf_split(s["csi"], s["w"], s["B"], s["U"], s["n"])
    else:
        m.zf(s["csi"], s["w"], s["B"], s["U"], s["n"])
    m.equalize_slots(s["w"], s["y"], s["llr"], **s["eq"])
    llr = s["llr"].view(torch.float16)
    # the mixed form's W is a private packing: its LLRs are the result
    return {"llr": llr} if s["form"] == m.FORM_MIXED else {"w": s["w"], "llr": llr}


def _graph(c, seed):
    n, lay = c["pushes"], _layout(c)
    G = _groups(c["N"], c["sg"])
    csi, y = _slot_inputs(c, seed, n)
    csi = csi.reshape(n, G, c["B"], c["U"])
    llr = torch.zeros(n, c["S"] * c["U"] * lay.ue_stride, dtype=torch.int16, device=DEV)
    g = pipeline.PipelineGraph([(csi[i], y[i], llr[i]) for i in range(n)], num_ue=c["U"],
                               num_bs=c["B"], num_sc=c["N"], sc_group=c["sg"],
                               num_syms=c["S"], mod_order=c["Q"], form=_form(c),
                               **_place(c, lay))
    return dict(kind="graph", g=g, llr=llr)


def _run_graph(s):
    s["g"].launch()
    return {"llr": s["llr"].view(torch.float16)}


def _batch_cells(c):
    return synth.uneven_cells(c["cells"], c["pick"])


def _batch_inputs(c, seed):
    for k, d in enumerate(_batch_cells(c)):
        yield d, *_slot_inputs(d, seed * 64 + k, 1)


def _batch(c, seed):
    cfgs = _batch_cells(c)
    lays = [synth.standalone_layout(d["N"], d["Q"]) for d in cfgs]
    nw = [_groups(d["N"], d["sg"]) * d["B"] * d["U"] for d in cfgs]
    nl = [d["S"] * d["U"] * lay.ue_stride for d, lay in zip(cfgs, lays)]
    w = torch.zeros(sum(nw), dtype=torch.complex64, device=DEV)
    llr = torch.zeros(sum(nl), dtype=torch.int16, device=DEV)
    cells = []
    for (d, csi, y), lay, wk, lk in zip(_batch_inputs(c, seed), lays, w.split(nw), llr.split(nl)):
        cells.append(dict(U=d["U"], B=d["B"], N=d["N"], sg=d["sg"], S=d["S"], Q=d["Q"],
                          layout=lay, csi=csi, y=y, w=wk, llr=lk))
    return dict(kind="batch", h=m.Batch(cells), w=w, llr=llr)


def _run_batch(s):
    s["h"].run()
    return {"w": s["w"], "llr": s["llr"].view(torch.float16)}


def _start(ca, N):
    return (ca - N) // 2


def _cols(ca, N):
    """FFT bin of subcarrier i."""
    return (torch.arange(N, device=DEV) + _start(ca, N) + ca // 2) % ca


def _samples(spec, bits):
    """Integer (re, im) samples of spectra spec [...][ca] at 40 % of full scale."""
    t = torch.fft.ifft(spec)
    r = torch.view_as_real(t)
    full = 32768 if bits == 16 else 128
    r = (r * (0.4 * full / r.abs().max())).round()
    return r.to(torch.int16 if bits == 16 else torch.int8).contiguous()


def _uplink_inputs(c, seed):
    """(pilot samples [P][B][ca][2], data samples [S][B][ca][2], pilot sign):
    pilot symbol p carries users p*sg .. p*sg + sg - 1 of every group."""
    U, B, ca, N, sg, S = (c[k] for k in ("U", "B", "ca", "N", "sg", "S"))
    G, P = _groups(N, sg), -(-U // sg)
    gen = _gen(seed)
    H = _channel(gen, G, B, U, "iid")
    y = _received(gen, H, 1, N, sg, S, c["Q"], c["snr"])[0]
    sign = torch.from_numpy(m.pilot_sign(N)).to(DEV)
    spec = torch.zeros(P + S, B, ca, dtype=torch.complex64, device=DEV)
    i, cols = torch.arange(N, device=DEV), _cols(ca, N)
    for p in range(P):
        u = p * sg + i % sg
        ok = u < U
        spec[p][:, cols[ok]] = (H[i[ok] // sg, :, u[ok]] / torch.conj(sign[ok])[:, None]).T
    spec[P:, :, cols] = y
    iq = _samples(spec, c["bits"])
    return iq[:P].contiguous(), iq[P:].contiguous(), sign


def _uplink(c, seed):
    U, B, ca, N, sg, S, Q = (c[k] for k in ("U", "B", "ca", "N", "sg", "S", "Q"))
    G, lay = _groups(N, sg), synth.standalone_layout(N, Q)
    pil, dat, sign = _uplink_inputs(c, seed)
    csi = torch.zeros(G, B, U, dtype=torch.complex64, device=DEV)
    up = m.UplinkDetect(ofdm_start=_start(ca, N), ofdm_ca=ca, ofdm_num=N, bs_num=B, num_syms=S,
                        quant_bits=c["bits"], num_ue=U, sc_group=sg, mod_order=Q,
                        **_place(c, lay))
    return dict(kind="uplink", pil=pil, dat=dat, sign=sign, csi=csi, w=torch.zeros_like(csi),
                llr=torch.zeros(S * U * lay.ue_stride, dtype=torch.int16, device=DEV), up=up,
                B=B, U=U, G=G, sg=sg,
                fft=dict(ofdm_start=_start(ca, N), ofdm_ca=ca, ofdm_num=N, bs_num=B))


def _run_uplink(s):
    m.pilot_fft(s["pil"], s["csi"], s["sign"], ue_num=s["U"], sc_group=s["sg"],
                num_syms=s["pil"].shape[0], **s["fft"])
    m.zf(s["csi"], s["w"], s["B"], s["U"], s["G"])
    s["up"].run(s["dat"], s["w"], s["llr"])
    return {"csi": s["csi"], "w": s["w"], "llr": s["llr"].view(torch.float16)}


def _precode_inputs(c, seed):
    """(W [G][B][U] of a CN(0, 1) channel, user symbols [S][U][N])."""
    gen = _gen(seed)
    A = _csi(_channel(gen, _groups(c["N"], c["sg"]), c["B"], c["U"], "iid"))
    w = _zf64(A).to(torch.complex64).contiguous()
    return w, _symbols(gen, 6, c["S"], c["U"], c["N"])


def _precode(c, seed):
    w, ue = _precode_inputs(c, seed)
    out = torch.zeros(c["S"], c["B"], c["ca"], dtype=torch.complex64, device=DEV)
    return dict(kind="precode", w=w, ue=ue, prec=torch.zeros_like(w), out=out, U=c["U"],
                B=c["B"], G=w.shape[0],
                kw=dict(num_bs=c["B"], num_ue=c["U"], num_sc=c["N"], sc_group=c["sg"],
                        bs_stride=c["ca"], bs_start=_start(c["ca"], c["N"]), num_syms=c["S"]))


def _run_precode(s):
    m.Beamform.beamform_downlink(s["w"], s["prec"], s["U"], s["B"], s["G"])
    m.precode(s["prec"], s["ue"], s["out"], **s["kw"])
    return {"precoder": s["prec"], "out": s["out"]}


def _ifft(c, seed):
    gen = _gen(seed)
    ca, N = c["ca"], c["N"]
    x = torch.zeros(c["S"], c["B"], ca, dtype=torch.complex64, device=DEV)
    # a tenth of full scale (RMS) after the transform, as a transmitter backs off
    x[:, :, _cols(ca, N)] = 0.1 * ca / math.sqrt(N) * _cn(gen, c["S"], c["B"], N)
    iq = torch.zeros(c["S"], c["B"], ca, 2, device=DEV,
                     dtype=torch.int16 if c["bits"] == 16 else torch.int8)
    return dict(kind="ifft", x=x, iq=iq, kw=dict(ofdm_ca=ca, bs_num=c["B"], num_syms=c["S"]))


def _run_ifft(s):
    m.downlink_ifft(s["x"], s["iq"], **s["kw"])
    return {"iq": s["iq"]}


def _ldpc(c, seed):
    """The all-zero codeword (a codeword of every linear code; the decoder is
    symmetric in the bits) through BPSK + AWGN, each block at an SNR of its
    own around the code's threshold, so that some blocks decode and some do
    not."""
    gen = _gen(seed)
    kb = 22 if c["bg"] == 1 else 10
    nv, words = (kb + c["mb"]) * c["zc"], (kb * c["zc"] + 31) // 32
    stride = synth.pad64(nv)
    rate = kb / (kb + c["mb"] - 2)
    snr = 10 * math.log10(rate) + 4.0 * torch.rand(c["cb"], 1, device=DEV, generator=gen)
    sigma = torch.sqrt(0.5 / 10.0 ** (snr / 10))
    llr = torch.zeros(c["cb"], stride, device=DEV)
    noise = torch.randn(c["cb"], nv, device=DEV, generator=gen)
    llr[:, :nv] = 2 * (1.0 + sigma * noise) / sigma ** 2
    llr[:, :2 * c["zc"]] = 0
    if c["bits"] == 16:
        llr = llr.to(torch.float16)
    out = torch.zeros(c["cb"], words, dtype=torch.int32, device=DEV)
    return dict(kind="ldpc", llr=llr, out=out,
                kw=dict(base_graph=c["bg"], lifting_size=c["zc"], parity_nodes=c["mb"],
                        max_iterations=c["iters"], num_cb=c["cb"], llr_stride=stride,
                        out_stride=words))


def _run_ldpc(s):
    m.ldpc_decode(s["llr"], s["out"], **s["kw"])
    return {"bits": s["out"]}


def _learned_inputs(c, seed):
    """CSI of two consecutive slots of a time-varying channel, and y of the
    second."""
    chan = learned.GpuChannel(synth.TdlJakes(c["B"], c["U"], c["N"], c["sg"], seed=seed))
    prev, cur = chan.slot(500), chan.slot(501)
    y = _received(_gen(seed), _csi(cur), 1, c["N"], c["sg"], c["S"], c["Q"], c["snr"])[0]
    return prev, cur, y


def _learned(c, seed):
    U, B, N, sg, S, Q = (c[k] for k in ("U", "B", "N", "sg", "S", "Q"))
    G, lay = _groups(N, sg), synth.standalone_layout(N, Q)
    prev, cur, y = _learned_inputs(c, seed)
    net, _ = learned.load(CKPT)
    z = learned.LearnedZF(U, B, G, net)
    z.step(prev)
    eq = dict(num_ue=U, num_bs=B, num_sc=N, sc_group=sg, num_syms=S, num_slots=1, mod_order=Q,
              csi_slot_stride=G * B * U, y_sym_stride=B * N, y_slot_stride=S * B * N,
              llr_sym_stride=U * lay.ue_stride, llr_slot_stride=S * U * lay.ue_stride,
              **_place(c, lay))
    return dict(kind="learned", z=z, cur=cur, y=y, eq=eq, first=z.k,
                llr=torch.zeros(S * U * lay.ue_stride, dtype=torch.int16, device=DEV))


def _run_learned(s):
    s["z"].k = s["first"]  # every pass starts from the previous slot's state
    w, info = s["z"].step(s["cur"])
    m.equalize_slots(w, s["y"], s["llr"], **s["eq"])
    return {"w": w, "info": info, "llr": s["llr"].view(torch.float16)}


def _train_inputs(c, seed):
    """Features (upper triangles of the scaled Gram difference and previous
    inverse) and targets (scaled error of the first-order update) of
    consecutive slots of a time-varying channel, in float64 on the host."""
    U, G = c["U"], c["G"]
    chan = learned.GpuChannel(synth.TdlJakes(c["B"], U, G * 12, 12, seed=seed))
    slots = [chan.slot(t).to(torch.complex128) for t in range(c["pairs"] + 1)]
    grams = [torch.matmul(a.transpose(1, 2).contiguous(), a.conj().resolve_conj()).cpu()
             for a in slots]
    inv = [torch.linalg.inv(g) for g in grams]
    iu = torch.triu_indices(U, U)
    tri = lambda t: torch.view_as_real(t[:, iu[0], iu[1]]).reshape(t.shape[0], -1)  # noqa: E731
    xs, ts = [], []
    for p in range(c["pairs"]):
        dg = grams[p + 1] - grams[p]
        s = grams[p].diagonal(dim1=1, dim2=2).real.mean(1)[:, None, None]
        base = inv[p] - inv[p] @ dg @ inv[p]
        xs.append(torch.cat([tri(dg / s), tri(inv[p] * s)], 1))
        ts.append(tri((inv[p + 1] - base) * s))
    return torch.cat(xs).to(torch.bfloat16), torch.cat(ts).float()


def _net(c, seed):
    return learned.WarmStartNet(c["U"], seed=seed)


def _train(c, seed):
    x, t = _train_inputs(c, seed)
    return dict(kind="train", net=_net(c, seed), x=x.to(DEV), t=t.to(DEV))


def _run_train(s):
    net = s["net"]
    out = net.forward(s["x"], keep=True)
    grads = net.backward(net.mse_grad(out, s["t"]))
    net.adam(lr=1e-3)
    return {"out": out, "grads": list(grads), "params": list(net.params)}


_PREPARE = dict(slots=_slots, graph=_graph, batch=_batch, uplink=_uplink, precode=_precode,
                ifft=_ifft, ldpc=_ldpc, learned=_learned, train=_train)
_RUN = dict(slots=_run_slots, graph=_run_graph, batch=_run_batch, uplink=_run_uplink,
            precode=_run_precode, ifft=_run_ifft, ldpc=_run_ldpc, learned=_run_learned,
            train=_run_train)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["kind"]](state)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _detect_work(U, B, N, sg, S, Q, slots=1, w_out=True, y=True):
    G = _groups(N, sg)
    byts = 8 * U * B * G * (2 if w_out else 1) + (8 * B * N * S if y else 0) + 2 * U * Q * N * S
    zf = G * (4 * U * (U + 1) * B + 8 * U * U * B + 4 / 3 * U ** 3)
    return slots * byts, slots * (zf + 8 * U * B * N * S)


def work(case):
    c = case
    kind = c["kind"]
    if kind in ("slots", "graph"):
        b, f = _detect_work(c["U"], c["B"], c["N"], c["sg"], c["S"], c["Q"],
                            c.get("slots") or c["pushes"], kind == "slots")
    elif kind == "batch":
        per = [_detect_work(d["U"], d["B"], d["N"], d["sg"], d["S"], d["Q"])
               for d in _batch_cells(c)]
        b, f = sum(p[0] for p in per), sum(p[1] for p in per)
    elif kind == "uplink":
        P = -(-c["U"] // c["sg"])
        b, f = _detect_work(c["U"], c["B"], c["N"], c["sg"], c["S"], c["Q"], y=False)
        b += (P + c["S"]) * c["B"] * c["ca"] * c["bits"] / 4
        f += (P + c["S"]) * c["B"] * 5 * c["ca"] * math.log2(c["ca"])
    elif kind == "precode":
        G = c["N"] // c["sg"]
        n = G * c["sg"] * c["S"]
        b = 8 * (2 * c["U"] * c["B"] * G + (c["U"] + c["B"]) * n)
        f = 8 * c["U"] * c["B"] * n
    elif kind == "ifft":
        n = c["S"] * c["B"]
        b, f = n * c["ca"] * (8 + c["bits"] / 4), n * 5 * c["ca"] * math.log2(c["ca"])
    elif kind == "ldpc":
        kb, edges = (22, 316) if c["bg"] == 1 else (10, 197)
        edges = edges * c["mb"] / (46 if c["bg"] == 1 else 42)
        b = c["cb"] * c["zc"] * ((kb + c["mb"] - 2) * c["bits"] / 8 + kb / 8)
        # a subtract, a compare of magnitudes, a scaling and an add per edge
        f = c["cb"] * c["iters"] * edges * c["zc"] * 4
    elif kind == "learned":
        b, f = _detect_work(c["U"], c["B"], c["N"], c["sg"], c["S"], c["Q"])
        d = [learned.n_features(c["U"]), 512, 512, learned.n_outputs(c["U"])]
        n = sum(d[i] * d[i + 1] for i in range(3))
        b += 2 * n
        f += 2 * _groups(c["N"], c["sg"]) * n
    else:
        d = [learned.n_features(c["U"]), 512, 512, learned.n_outputs(c["U"])]
        M, n = c["G"] * c["pairs"], sum(d[i] * d[i + 1] for i in range(3))
        # features, targets; FP32 weights, moments in and out, gradients out
        b = M * (2 * d[0] + 4 * d[3]) + n * (6 * 4 + 4)
        f = 2 * M * (3 * n - d[0] * d[1])
    return {"bytes": float(b), "flops": float(f)}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------

def _zf64(A):
    """W = (A A^H)^-1 A per group for A = csi^T: csi, W [G][B][U]."""
    a = A.to(torch.complex128)                       # [G][B][U]
    at = a.transpose(1, 2).contiguous()              # [G][U][B]
    gram = torch.matmul(at, a.conj().resolve_conj())
    x = torch.linalg.inv(gram.cpu()).to(a.device)
    return torch.matmul(x, at).transpose(1, 2).contiguous()


def _demod64(x, Q):
    """Max-log LLRs [..., Q] in units of the demod's scale."""
    re, im = x.real, x.imag
    if Q == 2:
        return torch.stack([re, im], -1) * (-20.0 * math.sqrt(2.0))
    ls = [100.0 * re, 100.0 * im]
    for t in {4: (200 / math.sqrt(10),), 6: (400 / math.sqrt(42), 200 / math.sqrt(42)),
              8: (800 / math.sqrt(170), 400 / math.sqrt(170), 200 / math.sqrt(170))}[Q]:
        ls += [t - ls[-2].abs(), t - ls[-1].abs()]
    return torch.stack(ls, -1)


def _llr64(W, y, N, sg, Q, lay):
    """LLR rows [S][U][ue_stride] of one slot: W [G][B][U], y [S][B][N]."""
    G, B, U = W.shape
    S = y.shape[0]
    yp = torch.zeros(S, B, G * sg, dtype=torch.complex128, device=y.device)
    yp[..., :N] = y
    yg = yp.reshape(S, B, G, sg).permute(2, 1, 0, 3).reshape(G, B, S * sg).contiguous()
    x = torch.matmul(W.transpose(1, 2).contiguous(), yg)
    x = x.reshape(G, U, S, sg).permute(2, 1, 0, 3).reshape(S, U, G * sg)[..., :N]
    bits = _demod64(x, Q).reshape(S, U, N * Q)
    k = torch.arange(N * Q, device=y.device)
    j = k % Q
    k0 = k - j
    at = k0 // lay.cb_size * lay.cb_stride + lay.zeros + k0 % lay.cb_size + j
    ok = (k < lay.valid_bits) & (at < lay.ue_stride)
    out = torch.zeros(S, U, lay.ue_stride, dtype=torch.float64, device=y.device)
    out[..., at[ok]] = bits[..., ok]
    return out


def _spectrum64(iq, ca, N):
    full = 32768.0 if iq.dtype == torch.int16 else 128.0
    x = torch.view_as_complex(iq.to(torch.float64) / full)
    return torch.fft.fft(x)[..., _cols(ca, N)]


def _exact_slots(c, seed):
    n = c.get("slots") or c["pushes"]
    csi, y = _slot_inputs(c, seed, n)
    W = _zf64(csi)
    G, lay = _groups(c["N"], c["sg"]), _layout(c)
    llr = torch.stack([_llr64(W[i * G:(i + 1) * G], y[i], c["N"], c["sg"], c["Q"], lay)
                       for i in range(n)])
    if c["kind"] == "graph":
        return {"llr": llr.reshape(n, -1)}
    return {"llr": llr.reshape(-1)} if c["form"] == "mixed" else \
        {"w": W.reshape(-1), "llr": llr.reshape(-1)}


def _exact_batch(c, seed):
    ws, ls = [], []
    for d, csi, y in _batch_inputs(c, seed):
        W = _zf64(csi)
        ws.append(W.reshape(-1))
        ls.append(_llr64(W, y[0], d["N"], d["sg"], d["Q"],
                         synth.standalone_layout(d["N"], d["Q"])).reshape(-1))
    return {"w": torch.cat(ws), "llr": torch.cat(ls)}


def _exact_uplink(c, seed):
    pil, dat, sign = _uplink_inputs(c, seed)
    U, B, ca, N, sg = (c[k] for k in ("U", "B", "ca", "N", "sg"))
    G = _groups(N, sg)
    csi = torch.zeros(G, B, U, dtype=torch.complex128, device=DEV)
    i = torch.arange(N, device=DEV)
    X = _spectrum64(pil, ca, N)
    for p in range(pil.shape[0]):
        u = p * sg + i % sg
        ok = u < U
        v = torch.conj(X[p][:, ok]) * sign[ok].to(torch.complex128)
        csi[i[ok] // sg, :, u[ok]] = v.T.contiguous()
    W = _zf64(csi)
    y = _spectrum64(dat, ca, N)
    return {"csi": csi, "w": W,
            "llr": _llr64(W, y, N, sg, c["Q"], synth.standalone_layout(N, c["Q"])).reshape(-1)}


def _exact_precode(c, seed):
    w, ue = _precode_inputs(c, seed)
    U, B, N, sg, S, ca = (c[k] for k in ("U", "B", "N", "sg", "S", "ca"))
    G, full = w.shape[0], N // sg
    w64 = w.to(torch.complex128)
    P = (w64 / w64.abs().amax((1, 2), keepdim=True)).transpose(1, 2).contiguous()   # [G][U][B]
    u = ue[..., :full * sg].to(torch.complex128).reshape(S, U, full, sg)
    u = u.permute(2, 1, 0, 3).reshape(full, U, S * sg).contiguous()
    x = torch.matmul(P[:full].transpose(1, 2).contiguous(), u)
    x = x.reshape(full, B, S, sg).permute(2, 1, 0, 3).reshape(S, B, full * sg)
    out = torch.zeros(S, B, ca, dtype=torch.complex128, device=DEV)
    out[:, :, _cols(ca, full * sg) if full * sg == N else
        (torch.arange(full * sg, device=DEV) + _start(ca, N) + ca // 2) % ca] = x
    return {"precoder": P.reshape(w.shape), "out": out}


def _exact_learned(c, seed):
    _, cur, y = _learned_inputs(c, seed)
    W = _zf64(cur)
    lay = synth.standalone_layout(c["N"], c["Q"])
    return {"w": W.reshape(-1), "info": None,
            "llr": _llr64(W, y, c["N"], c["sg"], c["Q"], lay).reshape(-1)}


def _exact_train(c, seed):
    """The step on the FP32 weights and BF16 features, without the rounding of
    weights and activations to BF16 inside."""
    x, t = (v.double() for v in _train_inputs(c, seed))
    net = _net(c, seed)
    par = [p.double().cpu().requires_grad_(True) for p in net.params]
    h = x
    for layer in range(3):
        h = h @ par[layer] + par[3 + layer]
        if layer < 2:
            h = torch.nn.functional.gelu(h, approximate="tanh")
    grads = torch.autograd.grad(0.5 * ((h - t) ** 2).sum() / h.shape[0], par)
    after = [p - 1e-3 * g / (g.abs() + 1e-8) for p, g in zip(par, grads)]
    return {"out": h.detach(), "grads": list(grads), "params": [p.detach() for p in after]}


_EXACT = dict(slots=_exact_slots, graph=_exact_slots, batch=_exact_batch, uplink=_exact_uplink,
              precode=_exact_precode, learned=_exact_learned, train=_exact_train)


def exact(case, seed):
    """None for the kinds whose outputs are whole numbers (IFFT, LDPC)."""
    f = _EXACT.get(case["kind"])
    return None if f is None else f(case, seed)
