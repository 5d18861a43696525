"""Causal chunks on the fp32-class chunk kernel (csrc/paged_prefill_split.hip):
fp32 K/V and the bf16 shapes the bf16 block kernel does not cover, at the
edges of its tiles (16-vector blocks, 32-key tiles, key splits), against the
oracle's restatement of PrefillAttentionVarlenF32 and against the same step
with every row on the decode kernels (EHIP_PREFILL=0; =1 keeps small chunks
beside a decode row on the chunk kernel).

Bars: 1e-4 relative per output vector against the fp32 oracle and the decode
kernels, their own bar; against 64 bits 5e-7 in the 2-norm, below what a plane
less of any operand costs (test_chunks_keep_the_third_planes): the products
left out of the plane splits are below 3 * 2^-24 of |q||k| (and |p||v|) per
term, sums are fp32 over at most a few thousand terms, and the hardware
exponential is within 2^-22 at these arguments."""
from types import SimpleNamespace

import numpy as np
import pytest

from gpu_util import rel_norm
from paged_util import scale_for

pytestmark = pytest.mark.gpu

BAR = 1e-4


def make_case(orc, bf16, H, Hkv, d, bs, chunks, seed):
    """Chunks (T, P) plus one decode row over a shuffled pool; poison outside."""
    rng = np.random.default_rng(seed)
    qlens = [t for t, _ in chunks] + [1]
    lens = [t + p for t, p in chunks] + [77]
    need = [-(-n // bs) for n in lens]
    pool = sum(need) + 3
    perm = rng.permutation(pool).astype(np.int32)
    tables, at = [], 0
    for n in need:
        tables.append(perm[at:at + n].copy())
        at += n
    k = np.full((pool, Hkv, bs, d), 1e30, np.float32)
    v = np.full_like(k, 1e30)
    ks, vs = [], []
    for t, n in zip(tables, lens):
        kk = rng.standard_normal((Hkv, n, d)).astype(np.float32)
        vv = rng.standard_normal((Hkv, n, d)).astype(np.float32)
        if bf16:
            kk = orc.bf16_bits_to_f32(orc.to_bf16_bits(kk))
            vv = orc.bf16_bits_to_f32(orc.to_bf16_bits(vv))
        for s in range(n):
            k[t[s // bs], :, s % bs] = kk[:, s]
            v[t[s // bs], :, s % bs] = vv[:, s]
        ks.append(kk)
        vs.append(vv)
    q = rng.standard_normal((sum(qlens), H, d)).astype(np.float32)
    return SimpleNamespace(bf16=bf16, H=H, Hkv=Hkv, d=d, bs=bs, qlens=qlens, lens=lens,
                           tables=tables, pool=pool, k=k, v=v, ks=ks, vs=vs, q=q)


def run(ctx, ehip_mod, orc, c, shift=0):
    """The step's outputs; shift moves every operand by that many bytes."""
    def up(a):
        b = ctx.alloc(a.nbytes + shift)
        raw = np.zeros(a.nbytes + shift, np.uint8)
        raw[shift:] = a.view(np.uint8).ravel()
        b.upload(raw)
        return b, SimpleNamespace(ptr=b.ptr + shift)

    k = orc.to_bf16_bits(c.k) if c.bf16 else c.k
    v = orc.to_bf16_bits(c.v) if c.bf16 else c.v
    bufs = [up(a) for a in (c.q, k, v, np.zeros_like(c.q))]
    dt = ehip_mod.KV_BF16 if c.bf16 else ehip_mod.KV_F32
    g = ehip_mod.geometry(c.H, c.Hkv, c.d, c.bs, dt, c.pool, scale_for(c.d))
    st = ehip_mod.StepArrays(c.qlens, c.lens, c.tables)
    assert ctx.step_upload(g, st) == 0, ctx.last_error()
    assert ctx.step_attention(*(p for _, p in bufs)) == 0, ctx.last_error()
    ctx.sync()
    raw = bufs[3][0].download(np.uint8, (c.q.nbytes + shift,))
    for b, _ in bufs:
        b.free()
    return raw[shift:].view(np.float32).reshape(c.q.shape)


def exact(q, ks, vs, qlens, lens, scale):
    """The chunks' attention in 64 bits: q [rows, H, d], per sequence K and V
    [Hkv, L, d]. Rows of a sequence sit at its last positions."""
    q = np.asarray(q, np.float64)
    H = q.shape[1]
    out, at = np.empty_like(q), 0
    for k, v, t, n in zip(ks, vs, qlens, lens):
        k = np.repeat(np.asarray(k, np.float64), H // k.shape[0], axis=0)
        v = np.repeat(np.asarray(v, np.float64), H // v.shape[0], axis=0)
        s = q[at:at + t].transpose(1, 0, 2) @ k.transpose(0, 2, 1) * scale
        s[:, np.arange(n)[None, :] > np.arange(n - t, n)[:, None]] = -np.inf
        p = np.exp(s - s.max(axis=2, keepdims=True))
        out[at:at + t] = ((p @ v) / p.sum(axis=2, keepdims=True)).transpose(1, 0, 2)
        at += t
    return out


def rel2(a, b):
    """2-norm of the difference over the 2-norm of b."""
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


def two_planes(x):
    """fp32 values cut to the two leading bf16 planes of three."""
    def rne(v):
        b = v.view(np.uint32)
        return ((b + 0x7FFF + (b >> 16 & 1)) & np.uint32(0xFFFF0000)).view(np.float32)

    x = np.ascontiguousarray(x, np.float32)
    hi = rne(x)
    return hi + rne(x - hi)


def reference(orc, c):
    cu = np.concatenate([[0], np.cumsum(c.qlens)]).astype(np.int32)
    return orc.prefill_varlen(c.q, cu, c.ks, c.vs, c.H, c.Hkv, c.d, scale_for(c.d), isa=1)


@pytest.mark.parametrize("bf16,H,Hkv,d,bs", [
    (False, 14, 2, 64, 16), (False, 14, 2, 64, 8), (False, 8, 8, 64, 64), (False, 32, 8, 128, 16),
    (False, 64, 1, 64, 16), (False, 6, 2, 128, 32), (True, 14, 2, 64, 16), (True, 8, 4, 128, 8),
    (True, 32, 8, 128, 8)])
@pytest.mark.parametrize("chunks", [[(16, 0), (17, 31)], [(33, 5), (130, 0)], [(40, 700)]],
                         ids=["edges", "ragged", "splits"])
def test_chunks_match_the_oracle(ehip_mod, orc, tctx, bf16, H, Hkv, d, bs, chunks):
    c = make_case(orc, bf16, H, Hkv, d, bs, chunks, seed=H + d + bs + chunks[0][0])
    ref = reference(orc, c)
    ctx = tctx(EHIP_PREFILL="1")
    got = run(ctx, ehip_mod, orc, c)
    assert rel_norm(got, ref) <= BAR, rel_norm(got, ref)
    if chunks[0][1] == 700:  # 24 tiles: cut into key splits
        assert ctx.step_info()[2] > 2 * Hkv
    rows = run(tctx(EHIP_PREFILL="0"), ehip_mod, orc, c)
    assert rel_norm(got, rows) <= BAR, rel_norm(got, rows)


@pytest.mark.parametrize("bf16,d", [(False, 64), (False, 128), (True, 64)])
def test_chunk_operands_at_any_alignment(tctx, ehip_mod, orc, bf16, d):
    """q, slabs and outputs 4 bytes off a 16-byte boundary, as the decode
    kernels take them (the decode row after the chunk takes another of them
    there)."""
    ctx = tctx(EHIP_PREFILL="1")
    c = make_case(orc, bf16, 14, 2, d, 16, [(45, 20)], seed=d)
    off, on = run(ctx, ehip_mod, orc, c, shift=4), run(ctx, ehip_mod, orc, c)
    assert np.array_equal(off[:45], on[:45])
    assert rel_norm(off, on) <= BAR


@pytest.mark.parametrize("bf16,d", [(False, 64), (False, 128), (True, 64)])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_rows_before_a_non_finite_value_stay_clean(tctx, ehip_mod, orc, bf16, d, bad):
    """A non-finite V element reaches the rows that attend its key, in its
    column, and no other output."""
    ctx = tctx(EHIP_PREFILL="1")
    c = make_case(orc, bf16, 14, 2, d, 16, [(70, 40)], seed=3 + d)
    clean = run(ctx, ehip_mod, orc, c)
    pos, col = 83, 9  # key 83 of the chunk's sequence: rows 43.. attend it
    c.v[c.tables[0][pos // 16], 1, pos % 16, col] = bad
    got = run(ctx, ehip_mod, orc, c)
    hit = np.zeros(got.shape, bool)
    hit[43:70, 7:, col] = True
    assert not np.isfinite(got[hit]).any()
    if not np.isnan(bad):
        assert (got[hit] == (np.inf if bad > 0 else -np.inf)).all()
    got[hit] = clean[hit] = 0.0
    assert rel_norm(got, clean) <= BAR


@pytest.mark.parametrize("bf16,d", [(False, 64), (False, 128), (True, 64)])
def test_keys_at_minus_infinity_take_no_part(tctx, ehip_mod, orc, bf16, d):
    """A K element of -inf against positive queries scores -inf: its key has
    probability 0, as one scored -1e30 in the reference."""
    ctx = tctx(EHIP_PREFILL="1")
    c = make_case(orc, bf16, 14, 2, d, 16, [(70, 40)], seed=5 + d)
    pos, col = 83, 9
    c.q[:, :, col] = np.abs(c.q[:, :, col]) + 0.1
    c.k[c.tables[0][pos // 16], 1, pos % 16, col] = -np.inf
    c.ks[0][1, pos, col] = -1e30
    got = run(ctx, ehip_mod, orc, c)
    assert rel_norm(got, reference(orc, c)) <= BAR


def scaled_codes(rng, fp8, shape):
    """Random INT8 codes, or E4M3 ones of finite values, as bytes; and the
    values they stand for."""
    if not fp8:
        codes = rng.integers(-127, 128, shape).astype(np.int8)
        return codes.view(np.uint8), codes.astype(np.float64)
    codes = rng.integers(0, 256, shape).astype(np.uint8)
    codes[(codes & 0x7F) == 0x7F] = 0
    return codes, e4m3(codes)


def e4m3(codes):
    c = codes.astype(np.int32)
    e, m = c >> 3 & 15, c & 7
    mag = np.where(e == 0, np.ldexp(m / 8.0, -6), np.ldexp(1 + m / 8.0, e - 7))
    mag = np.where((c & 0x7F) == 0x7F, np.nan, mag)
    return np.where(c & 0x80, -mag, mag)


def run_scaled(ctx, ehip_mod, fp8, H, Hkv, d, bs, T, P, seed, edit=None):
    """One chunk of T rows after P keys over INT8 or FP8 K/V with random codes
    and scales; edit(q, k, v, ks, vs) changes q, codes and scales first, the
    sequence's block j being block j of the slab. Returns the kernel's rows and
    q and the dequantised K and V [Hkv, L, d]."""
    rng = np.random.default_rng(seed)
    L = T + P
    nb = -(-L // bs)
    q = rng.standard_normal((T, H, d)).astype(np.float32)
    k, v = (scaled_codes(rng, fp8, (nb, Hkv, bs, d))[0] for _ in "kv")
    top = 448.0 if fp8 else 127.0
    ks, vs = ((rng.uniform(1.5, 3.5, (nb, Hkv)) / top).astype(np.float32) for _ in "kv")
    if edit:
        edit(q, k, v, ks, vs)

    def values(codes, sc):
        x = e4m3(codes) if fp8 else codes.view(np.int8).astype(np.float64)
        with np.errstate(invalid="ignore"):
            x = x * sc.astype(np.float64)[:, :, None, None]
        return x.transpose(1, 0, 2, 3).reshape(Hkv, nb * bs, d)[:, :L]

    bufs = [ctx.to_device(x) for x in (q, k, v, ks, vs)] + [ctx.alloc(q.nbytes)]
    fmt = "fp8" if fp8 else "int8"
    dt = ehip_mod.KV_FP8 if fp8 else ehip_mod.KV_INT8
    g = ehip_mod.geometry(H, Hkv, d, bs, dt, nb, scale_for(d))
    st = ehip_mod.StepArrays([T], [L], [np.arange(nb, dtype=np.int32)])
    assert ctx.step_upload(g, st) == 0, ctx.last_error()
    assert getattr(ctx, "step_attention_" + fmt)(*bufs) == 0, ctx.last_error()
    ctx.sync()
    got = bufs[-1].download(np.float32, q.shape)
    for b in bufs:
        b.free()
    return got, q, values(k, ks), values(v, vs)


@pytest.mark.parametrize("M", [1e3, 1e5, 1e30])
@pytest.mark.parametrize("T,P", [(33, 64), (40, 700)], ids=["whole", "splits"])
@pytest.mark.parametrize("kv,d", [("f32", 64), ("f32", 128), ("bf16", 64), ("int8", 128),
                                  ("int8", 64), ("fp8", 128), ("fp8", 64)])
def test_scores_that_jump_between_tiles(tctx, ehip_mod, orc, kv, d, T, P, M):
    """A row's first 64 keys score about -M, its others as usual: the softmax
    reference jumps by M at its third tile, and the scores there keep their
    differences. Bars against 64 bits: 2e-6 (planes of 24 bits: about 2^-21 in
    a score of a few units, as far in a probability); over FP8 q has two planes,
    2^-18 of |q||k| is left out, 2e-5."""
    ctx = tctx(EHIP_PREFILL="1")
    low = -M / scale_for(d)
    if kv in ("f32", "bf16"):
        c = make_case(orc, kv == "bf16", 14, 2, d, 16, [(T, P)], seed=d + T)
        c.q[:T, :, 0] = 1.0
        c.ks[0][:, :, 0] = 0.0
        c.ks[0][:, :64, 0] = low
        if kv == "bf16":
            c.ks[0] = orc.bf16_bits_to_f32(orc.to_bf16_bits(c.ks[0]))
        for s in range(T + P):
            c.k[c.tables[0][s // 16], :, s % 16] = c.ks[0][:, s]
        got = run(ctx, ehip_mod, orc, c)[:T]
        ref = exact(c.q[:T], c.ks[:1], c.vs[:1], [T], [T + P], scale_for(d))
    else:
        def edit(q, k, v, ks, vs):
            q[:, :, 0] = 1.0
            k[:, :, :, 0] = 0
            k[:4] = 0
            k[:4, :, :, 0] = 0xFE if kv == "fp8" else 0x81  # -448, -127
            ks[:4] = -low / (448.0 if kv == "fp8" else 127.0)

        got, q, k, v = run_scaled(ctx, ehip_mod, kv == "fp8", 8, 2, d, 16, T, P, d + T, edit)
        ref = exact(q, [k], [v], [T], [T + P], scale_for(d))
    bar = 2e-5 if kv == "fp8" else 2e-6
    assert rel_norm(got, ref) <= bar, rel_norm(got, ref)


@pytest.mark.parametrize("bf16,d", [(False, 64), (False, 128), (True, 64)])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_non_finite_keys_reach_only_their_rows(tctx, ehip_mod, orc, bf16, d, bad):
    """A K element of +inf against positive queries, or NaN: the rows that
    attend its key have no finite output, the others are untouched."""
    ctx = tctx(EHIP_PREFILL="1")
    c = make_case(orc, bf16, 14, 2, d, 16, [(70, 40)], seed=7 + d)
    pos, col = 83, 9
    c.q[:, :, col] = np.abs(c.q[:, :, col]) + 0.1
    clean = run(ctx, ehip_mod, orc, c)
    c.k[c.tables[0][pos // 16], 1, pos % 16, col] = bad
    got = run(ctx, ehip_mod, orc, c)
    assert not np.isfinite(got[43:70, 7:]).any()
    got[43:70, 7:] = clean[43:70, 7:]
    assert rel_norm(got, clean) <= BAR


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("bad", [3.4e38, -3.4e38, float(np.finfo(np.float32).max)])
def test_values_past_the_bf16_range_stay_whole(tctx, ehip_mod, orc, d, bad):
    """fp32 values that round to infinity in bf16. As V of a key scored about
    -20 they arrive to 1e-5 (2^-21 |score| in the probability); as K against
    positive (bad < 0) or negative queries their key has probability 0."""
    ctx = tctx(EHIP_PREFILL="1")
    c = make_case(orc, False, 14, 2, d, 16, [(70, 40)], seed=9 + d)
    pos, col = 83, 9
    sign = -np.sign(bad)
    c.q[:, :, 3] = 1.0
    c.q[:, :, col] = sign * (np.abs(c.q[:, :, col]) + 0.1)
    c.ks[0][1, pos] = 0.0
    c.ks[0][1, pos, 3] = -20.0 / scale_for(d)
    c.vs[0][1, pos, col] = bad
    at = (c.tables[0][pos // 16], 1, pos % 16)
    c.k[at], c.v[at] = c.ks[0][1, pos], c.vs[0][1, pos]
    got = run(ctx, ehip_mod, orc, c)[:70]
    ref = exact(c.q[:70], c.ks[:1], c.vs[:1], [70], [110], scale_for(d))
    big = np.zeros(got.shape, bool)
    big[43:, 7:, col] = True
    assert (np.abs(got[big] - ref[big]) <= 1e-5 * np.abs(ref[big])).all()
    got[big] = ref[big] = 0.0
    assert rel_norm(got, ref) <= 1e-5

    c.ks[0][1, pos, col] = bad
    c.vs[0][1, pos, col] = 1.0
    c.k[at], c.v[at] = c.ks[0][1, pos], c.vs[0][1, pos]
    got = run(ctx, ehip_mod, orc, c)[:70]
    c.ks[0][1, pos] = 0.0
    c.ks[0][1, pos, 3] = -1e30
    ref = exact(c.q[:70], c.ks[:1], c.vs[:1], [70], [110], scale_for(d))
    assert rel_norm(got, ref) <= 1e-5


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("fp8,what", [
    (fp8, w) for fp8 in (False, True) for w in ("v_scale_inf", "v_scale_nan", "k_scale_nan")
] + [(True, "v_code_nan"), (True, "k_code_nan")])
def test_non_finite_scaled_kv_reaches_only_its_rows(tctx, ehip_mod, fp8, d, what):
    """A non-finite scale of a block, or a NaN code, that only the later rows
    attend: those rows have no finite output (of a V code: in its column), the
    earlier ones and the other kv heads are untouched."""
    ctx = tctx(EHIP_PREFILL="1")
    H, Hkv, T, P, pos, col = 8, 2, 70, 42, 96, 9  # position 96 opens block 6: rows 54..
    clean = run_scaled(ctx, ehip_mod, fp8, H, Hkv, d, 16, T, P, d)[0]

    def edit(q, k, v, ks, vs):
        if what == "v_code_nan":
            v[pos // 16, 1, 0, col] = 0xFF
        elif what == "k_code_nan":
            k[pos // 16, 1, 0, col] = 0x7F
        else:
            sc = vs if what[0] == "v" else ks
            sc[pos // 16, 1] = np.inf if what.endswith("inf") else np.nan

    got = run_scaled(ctx, ehip_mod, fp8, H, Hkv, d, 16, T, P, d, edit)[0]
    hit = np.zeros(got.shape, bool)
    hit[pos - P:, 4:, col if what == "v_code_nan" else slice(None)] = True
    assert not np.isfinite(got[hit]).any()
    got[hit] = clean[hit]
    assert rel_norm(got, clean) <= BAR


@pytest.mark.parametrize("kv,H,Hkv,d", [("f32", 14, 2, 64), ("f32", 32, 8, 128),
                                        ("bf16", 14, 2, 64), ("int8", 8, 2, 64),
                                        ("int8", 32, 8, 128), ("fp8", 8, 2, 64),
                                        ("fp8", 32, 8, 128)])
@pytest.mark.parametrize("T,P", [(90, 5), (40, 700)], ids=["whole", "splits"])
def test_chunks_keep_the_third_planes(tctx, ehip_mod, orc, kv, H, Hkv, d, T, P):
    """Error against 64 bits, below what an operand cut to two planes costs
    (about 2^-18 of it): 5e-7 in the 2-norm. FP8 takes q in two planes, 5e-6, as
    the decode kernels do; a plane less would cost 2^-9."""
    ctx = tctx(EHIP_PREFILL="1")
    if kv in ("f32", "bf16"):
        c = make_case(orc, kv == "bf16", H, Hkv, d, 16, [(T, P)], seed=T + d)
        q, k, v = c.q[:T], c.ks[0], c.vs[0]
        got = run(ctx, ehip_mod, orc, c)[:T]
    else:
        got, q, k, v = run_scaled(ctx, ehip_mod, kv == "fp8", H, Hkv, d, 16, T, P, T + d)
    ref = exact(q, [k], [v], [T], [T + P], scale_for(d))
    bar = 5e-6 if kv == "fp8" else 5e-7
    if kv != "fp8":  # the bar lies below the error of two planes
        assert rel2(exact(two_planes(q), [k], [v], [T], [T + P], scale_for(d)), ref) > bar
    if kv == "f32":
        assert rel2(exact(q, [two_planes(k)], [v], [T], [T + P], scale_for(d)), ref) > bar
        assert rel2(exact(q, [k], [two_planes(v)], [T], [T + P], scale_for(d)), ref) > bar
    assert rel2(got, ref) <= bar, rel2(got, ref)
