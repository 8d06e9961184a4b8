"""The LDPC consumer (mega_ldpc_decode) on cuda:0: the reference's decoder
test (test/ldpc/test_ldpc.cc:155-190: noiseless LLRs of encode.data decode to
input.data, one code block and two), bit-identical to the oracle's layered
min-sum on noisy code blocks of both base graphs (binary16 and float LLRs,
padded strides), and the chain the decoder exists for: LLRs of the
equalizer's LDPC layout (zeros = 2 * Zc, cb_size = (22 - 2 + mb) * Zc,
128-byte padded rows) decoded back into the transmitted information bits."""
import numpy as np
import pytest

import megastation_amd as m
from megastation_amd import synth
from oracle import ldpc

from gpu_helpers import dev_c64, make_slots, torch

pytestmark = pytest.mark.gpu


def _decode_gpu(llr_np, bg, zc, mb, iters, half, n_cb, llr_stride, out_stride, alpha=0.0):
    t = torch()
    dt = t.float16 if half else t.float32
    llr = t.from_numpy(llr_np.astype(np.float16 if half else np.float32).reshape(-1)).to("cuda:0")
    out = t.full((n_cb * out_stride,), -1, dtype=t.int32, device="cuda:0")
    m.ldpc_decode(llr.to(dt), out, base_graph=bg, lifting_size=zc, parity_nodes=mb,
                  max_iterations=iters, num_cb=n_cb, llr_stride=llr_stride,
                  out_stride=out_stride, normalization=alpha)
    t.cuda.synchronize()
    return out.cpu().numpy().view(np.uint32).reshape(n_cb, out_stride)


@pytest.mark.parametrize("half", [False, True])
def test_reference_codewords_decode_to_input_data(golden, half):
    print(f"case: ldpc reference fixture half={half}", flush=True)
    zc, mb = 64, 46
    enc = np.unpackbits(golden["ldpc_encoded_bits"], bitorder="little").reshape(2, 66 * zc)
    llr = np.zeros((2, 68 * zc), np.float32)
    llr[:, 2 * zc:] = np.where(enc == 1, -127.0, 127.0)
    words = 22 * zc // 32
    for n in (1, 2):                                # LDPCDecoderVec and LDPCDecoderArr
        out = _decode_gpu(llr[:n], 1, zc, mb, 8, half, n, 68 * zc, words)
        got = out.view(np.uint8).reshape(-1)
        assert np.array_equal(got, golden["ldpc_input_bits"][:n * 176])


@pytest.mark.parametrize("bg,zc,mb,half", [(1, 64, 46, False), (1, 288, 46, True),
                                           (2, 52, 42, False), (2, 384, 12, True),
                                           (1, 15, 4, False)])
def test_decoder_matches_oracle_on_noisy_code_blocks(bg, zc, mb, half):
    """Noise at a level the decoder only partly corrects in 4 iterations, so
    the comparison covers messages of both signs and unfinished decodes."""
    print(f"case: ldpc vs oracle bg={bg} zc={zc} mb={mb} half={half}", flush=True)
    kb = ldpc.KB[bg]
    n_cb = 5
    rng = np.random.default_rng(zc * 7 + mb)
    info = rng.integers(0, 2, (n_cb, kb * zc)).astype(np.uint8)
    cws = np.stack([ldpc.encode(b, bg, zc, mb) for b in info])
    sigma = 1.0
    llr = ((2 * ((1 - 2.0 * cws) + sigma * rng.standard_normal(cws.shape))) / sigma ** 2)
    llr[:, :2 * zc] = 0
    if half:
        llr = llr.astype(np.float16)
    llr = llr.astype(np.float32)                    # exactly what the kernel reads
    nv = (kb + mb) * zc
    stride = synth.pad64(nv)                        # 128-byte rows, like the equalizer's
    buf = np.zeros((n_cb, stride), np.float32)
    buf[:, :nv] = llr
    words = (kb * zc + 31) // 32
    out = _decode_gpu(buf, bg, zc, mb, 4, half, n_cb, stride, words + 3)
    ref = ldpc.decode(llr, bg, zc, mb, 4, 0.8125)
    assert np.array_equal(out[:, :words], ref)
    assert np.all(out[:, words:] == 0xFFFFFFFF)     # nothing written past the bits
    errs = (ldpc.unpack_bits(ref, kb * zc) != info).sum()
    print(f"  residual bit errors after 4 iterations: {errs}", flush=True)


@pytest.mark.parametrize("bg,zc,mb,half,n_cb", [(1, 288, 46, True, 257), (1, 384, 18, False, 258),
                                                (2, 320, 42, True, 259), (2, 256, 42, True, 257)])
def test_more_code_blocks_than_cus_match_oracle(bg, zc, mb, half, n_cb):
    """More code blocks than the card has CUs: from Zc > 256 on two of them share
    a workgroup where LDS holds both (the last may be alone). Five different
    blocks in turn, so that each meets each as its neighbour; bits and the padding
    after them are equal to the oracle's."""
    print(f"case: ldpc pairs bg={bg} zc={zc} mb={mb} half={half} n_cb={n_cb}", flush=True)
    kb = ldpc.KB[bg]
    rng = np.random.default_rng(zc + mb)
    info = rng.integers(0, 2, (5, kb * zc)).astype(np.uint8)
    cws = np.stack([ldpc.encode(b, bg, zc, mb) for b in info])
    llr = 2 * ((1 - 2.0 * cws) + rng.standard_normal(cws.shape))
    llr[:, :2 * zc] = 0
    llr = llr.astype(np.float16 if half else np.float32).astype(np.float32)
    nv, words = (kb + mb) * zc, (kb * zc + 31) // 32
    stride = synth.pad64(nv)
    buf = np.zeros((n_cb, stride), np.float32)
    turn = np.arange(n_cb) % 5
    buf[:, :nv] = llr[turn]
    out = _decode_gpu(buf, bg, zc, mb, 4, half, n_cb, stride, words + 1)
    ref = ldpc.decode(llr, bg, zc, mb, 4, 0.8125)
    assert np.array_equal(out[:, :words], ref[turn])
    assert np.all(out[:, words:] == 0xFFFFFFFF)


@pytest.mark.parametrize("bg,zc,mb", [(1, 72, 4), (1, 60, 24), (1, 60, 25), (2, 72, 4),
                                      (2, 60, 12), (2, 60, 13)])
def test_instances_for_few_rows_match_oracle(bg, zc, mb):
    """Either side of the row counts up to which a smaller instance decodes."""
    test_decoder_matches_oracle_on_noisy_code_blocks(bg, zc, mb, False)


@pytest.mark.parametrize("bg,zc,mb", [(1, 320, 24), (2, 288, 12), (2, 288, 5)])
def test_instances_for_few_rows_in_pairs_match_oracle(bg, zc, mb):
    test_more_code_blocks_than_cus_match_oracle(bg, zc, mb, True, 259)


def _decode_numpy(llr, bg, zc, mb, iters, alpha):
    """The layered schedule in numpy FP32 with the kernel's rule for NaN: not
    negative, never the minimum, min2 down to min1 (llr [n][(kb + mb) * zc])."""
    rs, col, shift = ldpc.tables(bg)
    sh, n, f32 = shift[ldpc.set_index(zc)], len(llr), np.float32
    L = llr.reshape(n, -1, zc).copy()
    R = np.zeros((rs[mb], n, zc), f32)
    for _ in range(iters):
        for r in range(mb):
            es = range(rs[r], rs[r + 1])
            q = [np.roll(L[:, col[e]], -(sh[e] % zc), axis=1) - R[e] for e in es]
            min1 = np.full((n, zc), np.inf, f32)
            min2, at, par = min1.copy(), np.zeros((n, zc), int), np.zeros((n, zc), bool)
            for i, x in enumerate(q):
                a = np.abs(x)
                at[a < min1] = i
                min2 = np.where(np.isnan(a), min1, np.maximum(min1, np.fmin(min2, a)))
                min1 = np.fmin(min1, a)
                par ^= x < 0
            for i, (e, x) in enumerate(zip(es, q)):
                mag = f32(alpha) * np.where(at == i, min2, min1)
                R[e] = np.where(par ^ (x < 0), -mag, mag)
                L[:, col[e]] = np.roll(x + R[e], sh[e] % zc, axis=1)
    bits = (L.reshape(n, -1)[:, :ldpc.KB[bg] * zc] < 0).astype(np.uint8)
    pad = np.zeros((n, -bits.shape[1] % 32), np.uint8)
    return np.packbits(np.hstack([bits, pad]), axis=1, bitorder="little").view(np.uint32)


@pytest.mark.parametrize("bg,zc,mb,half,n_cb", [(1, 288, 46, True, 258), (1, 64, 46, False, 5),
                                                (2, 384, 12, False, 257), (2, 15, 42, True, 5)])
@pytest.mark.filterwarnings("ignore:invalid value")
def test_infinite_and_nan_llrs(bg, zc, mb, half, n_cb):
    """Infinities of both signs (some cancel within a row) and NaN of both
    signs, one and two code blocks a workgroup: the bits of the same schedule in
    numpy, which agrees with the oracle where everything is finite."""
    print(f"case: ldpc non-finite bg={bg} zc={zc} mb={mb} half={half} n_cb={n_cb}", flush=True)
    nv, words = (ldpc.KB[bg] + mb) * zc, (ldpc.KB[bg] * zc + 31) // 32
    rng = np.random.default_rng(zc + 1)
    dt, it, nan = ((np.float16, np.uint16, (0x7e00, 0xfe00)) if half else
                   (np.float32, np.uint32, (0x7fc00000, 0xffc00000)))
    finite = rng.standard_normal((5, nv)).astype(dt)
    assert np.array_equal(_decode_numpy(finite.astype(np.float32), bg, zc, mb, 2, 0.8125),
                          ldpc.decode(finite.astype(np.float32), bg, zc, mb, 2, 0.8125))
    t = torch()
    turn = np.arange(n_cb) % 5
    for p_inf, p_nan in ((0.02, 0.0), (0.0, 0.002), (0.3, 0.05)):
        llr = finite.copy()
        u = rng.random(llr.shape)
        inf = u < p_inf
        llr[inf] = np.where(rng.random(inf.sum()) < 0.5, np.inf, -np.inf)
        isnan = u > 1 - p_nan
        llr.view(it)[isnan] = np.array(nan, it)[rng.integers(0, 2, isnan.sum())]
        dev = t.from_numpy(llr.view(np.int16 if half else np.int32)[turn]).to("cuda:0")
        for iters, alpha in ((1, 0.0), (3, 1.0)):  # 0 selects 0.8125
            out = t.zeros(n_cb, words, dtype=t.int32, device="cuda:0")
            m.ldpc_decode(dev.view(t.float16 if half else t.float32), out, base_graph=bg,
                          lifting_size=zc, parity_nodes=mb, max_iterations=iters, num_cb=n_cb,
                          llr_stride=nv, out_stride=words, normalization=alpha)
            ref = _decode_numpy(llr.astype(np.float32), bg, zc, mb, iters, alpha or 0.8125)
            assert np.array_equal(out.cpu().numpy().view(np.uint32), ref[turn]), (p_inf, iters)


def test_equalizer_llrs_decode_to_transmitted_bits():
    """64 x 16 cell, 1200 subcarriers, 16-QAM at -4 dB per antenna (about
    13 dB after ZF's array gain; the hard decisions of about 2 % of the coded
    bits are wrong): each user's symbol carries one rate-1/3 BG1 code block
    (Zc = 72: 22 * 72 <= 1200 * 4 / 3); ZF + equalize write its LLRs into the
    decoder's layout; the decoder gives back every information bit."""
    print("case: ldpc chain equalize -> decode", flush=True)
    t = torch()
    U, B, N, sg, Q, S, snr = 16, 64, 1200, 16, 4, 2, -4.0
    G = N // sg
    lay = synth.ldpc_uplink_layout(N, Q)
    zc = lay.zeros // 2
    mb = lay.cb_size // zc - 20
    assert (zc, mb) == (72, 46)
    rng = np.random.default_rng(11)
    info = rng.integers(0, 2, (S, U, 22 * zc)).astype(np.uint8)
    bits = rng.integers(0, 2, (S, U, N * Q)).astype(np.uint8)   # filler past cb_size
    for s in range(S):
        for u in range(U):
            bits[s, u, :lay.cb_size] = ldpc.encode(info[s, u], 1, zc, mb)[2 * zc:]
    sl = make_slots(5, 1, U, B, N, sg, S, Q, snr)[0]
    # the same channel and noise draw as make_slots, with these bits
    x = synth.modulate(bits.reshape(S, U, N, Q)).astype(np.complex64)
    Hk = sl.H[np.arange(N) // sg]
    y = np.einsum("kbu,suk->sbk", Hk, x).astype(np.complex64)
    y += (sl.y - np.einsum("kbu,suk->sbk", Hk, sl.x)).astype(np.complex64)   # its noise
    w = t.zeros(G * B * U, dtype=t.complex64, device="cuda:0")
    m.zf(dev_c64(sl.csi), w, B, U, G)
    llr = t.zeros(S * U * lay.ue_stride, dtype=t.int16, device="cuda:0")   # zero prefix
    m.equalize_slots(w, dev_c64(y), llr, num_ue=U, num_bs=B, num_sc=N, sc_group=sg,
                     num_syms=S, num_slots=1, mod_order=Q, ue_stride=lay.ue_stride,
                     cb_size=lay.cb_size, cb_stride=lay.cb_stride, zeros=lay.zeros,
                     valid_bits=lay.valid_bits, csi_slot_stride=G * B * U,
                     y_sym_stride=B * N, y_slot_stride=S * B * N,
                     llr_sym_stride=U * lay.ue_stride, llr_slot_stride=S * U * lay.ue_stride)
    words = 22 * zc // 32 + (1 if (22 * zc) % 32 else 0)
    out = t.zeros(S * U * words, dtype=t.int32, device="cuda:0")
    m.ldpc_decode(llr.view(t.float16), out, base_graph=1, lifting_size=zc, parity_nodes=mb,
                  max_iterations=8, num_cb=S * U, llr_stride=lay.cb_stride, out_stride=words)
    t.cuda.synchronize()
    dec = ldpc.unpack_bits(out.cpu().numpy().view(np.uint32).reshape(S * U, words), 22 * zc)
    raw = np.array(llr.cpu().numpy().view(np.float16), dtype=np.float32).reshape(
        S * U, lay.cb_stride)[:, lay.zeros:lay.zeros + lay.cb_size]
    raw_err = int(((raw < 0) != bits.reshape(S * U, -1)[:, :lay.cb_size]).sum())
    print(f"  channel bit errors before decoding: {raw_err}", flush=True)
    assert raw_err > 0                               # the decoder has work to do
    assert np.array_equal(dec, info.reshape(S * U, -1))


def test_ldpc_rejects_bad_arguments():
    print("case: ldpc argument checks", flush=True)
    t = torch()
    llr = t.zeros(68 * 64, dtype=t.float32, device="cuda:0")
    out = t.zeros(64, dtype=t.int32, device="cuda:0")
    kw = dict(base_graph=1, lifting_size=64, parity_nodes=46, max_iterations=8, num_cb=1,
              llr_stride=68 * 64, out_stride=44)
    m.ldpc_decode(llr, out, **kw)
    for bad, code in ((dict(base_graph=3), m.MEGA_ERR_UNSUPPORTED),
                      (dict(lifting_size=100), m.MEGA_ERR_UNSUPPORTED),
                      (dict(parity_nodes=47), m.MEGA_ERR_UNSUPPORTED),
                      (dict(max_iterations=0), m.MEGA_ERR_UNSUPPORTED),
                      (dict(llr_stride=68 * 64 - 1), m.MEGA_ERR_INVALID_ARG),
                      (dict(out_stride=43), m.MEGA_ERR_INVALID_ARG)):
        with pytest.raises(m.MegaError) as e:
            m.ldpc_decode(llr, out, **dict(kw, **bad))
        assert e.value.code == code, bad
