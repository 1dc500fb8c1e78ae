"""The many-row product (qdec_gemm from 9 rows at four waves, qdec_gemm_wide up
to 128) against the calls of at most 8 rows, bit for bit: every role's
epilogue, row counts at the edges of the row tiles, widths that leave a
workgroup short of output units and k ranges shorter than, equal to and past
its load ring."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def lib():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a HIP device")
    from qdec import capi
    return capi.lib()


def stream():
    return torch.cuda.current_stream().cuda_stream


def rnd(*shape, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16).to(DEV)


def pack(lib, w):
    dst = torch.empty(w.numel(), dtype=torch.bfloat16, device=DEV)
    lib.pack_tiles(w.data_ptr(), dst.data_ptr(), w.shape[0], w.shape[1], stream())
    return dst


def to_frag(x):
    """[rows, k] in fragment order, rows past the last NaN (they must not matter)."""
    rows, k = x.shape
    mt = -(-rows // 16)
    full = torch.full((mt * 16, k), float("nan"), dtype=torch.bfloat16, device=DEV)
    full[:rows] = x
    return full.view(mt, 16, k // 32, 4, 8).permute(2, 0, 3, 1, 4).contiguous()


def from_frag(buf, rows, cols):
    mt = -(-rows // 16)
    return buf.view(cols // 32, mt, 4, 16, 8).permute(1, 3, 0, 2, 4).reshape(mt * 16, cols)[:rows]


class Call:
    """One product in every form: kind -> the outputs of the rows given."""

    def __init__(self, lib, kind, n, k, ksplit, seed):
        from qdec import capi
        self.lib, self.capi, self.kind, self.n, self.k, self.ksplit = lib, capi, kind, n, k, ksplit
        glu = kind == "glu"
        self.w = pack(lib, rnd(2 * n if glu else n, k, scale=0.05, seed=seed))
        self.norm_w = rnd(k, scale=0.2, seed=seed + 1)
        self.scratch = torch.zeros(4 << 20, dtype=torch.float32, device=DEV)
        self.counters = torch.zeros(8192, dtype=torch.int32, device=DEV)
        self.waves, self.row_major, self.tiles, self.x_parts = 4, False, 1, None

    def __call__(self, x, res, wide):
        c, rows, n = self.capi, x.shape[0], self.n
        a = c.GemmArgs()
        flags = {"norm": c.NORM_IN, "glu": c.NORM_IN | c.GLU, "plain": 0, "res": c.RES_OUT, "parts": c.RES_OUT,
                 "argmax": c.NORM_IN | c.ARGMAX}[self.kind]
        a.w, a.eps, a.rows, a.n, a.k, a.flags = self.w.data_ptr(), 1e-6, rows, n, self.k, flags
        a.ksplit, a.waves, a.tiles_per_wg = self.ksplit, self.waves, self.tiles
        a.partial, a.counters = self.scratch.data_ptr(), self.counters.data_ptr()
        if flags & c.NORM_IN:
            a.x, a.norm_w = x.data_ptr(), self.norm_w.data_ptr()
            if self.x_parts is not None:
                self.merged = torch.full_like(x, float("nan"))
                a.x_parts, a.x_nparts, a.x_merged = (self.x_parts.data_ptr(), len(self.x_parts), self.merged.data_ptr())
        elif self.row_major:
            a.x = x.data_ptr()
        else:
            xf = to_frag(x)
            a.x, a.x_frag = xf.data_ptr(), 1
        mt = -(-rows // 16)
        out = torch.full((mt * 16, n), float("nan"), dtype=torch.bfloat16, device=DEV)
        r = res.clone()
        parts = torch.full((self.ksplit, rows, n), float("nan"), device=DEV)
        ids = torch.full((rows,), -1, dtype=torch.int64, device=DEV)
        lens = torch.zeros(rows, dtype=torch.int32, device=DEV)
        frag = self.kind == "glu" and n % 32 == 0
        if self.kind in ("norm", "glu", "plain", "argmax"):
            a.out, a.out_frag = out.data_ptr(), int(frag)
        else:
            a.res = r.data_ptr()
        if self.kind == "parts":
            a.parts_out = parts.data_ptr()
        if self.kind == "argmax":
            a.ids_out, a.lens_inc = ids.data_ptr(), lens.data_ptr()
        need = self.lib.gemm_wide_workspace(a) if wide else self.lib.gemm_workspace(a)[0]
        assert need <= self.scratch.numel() * 4
        (self.lib.gemm_wide if wide else self.lib.gemm)(a, stream())
        torch.cuda.synchronize()
        assert int(self.counters.abs().sum()) == 0
        if self.kind == "argmax":
            assert (lens == 1).all()
            return [out[:rows], ids]
        if self.kind == "parts":
            assert torch.equal(r, res)
            return list(parts)
        if self.kind == "res":
            return [r]
        return [from_frag(out, rows, n) if frag else out[:rows]]


# (kind, n, k, ksplit): one output unit and one k step per wave; units that do
# not divide among workgroups; more units than one round of three; k splits.
SHAPES = [("norm", 16, 128, 1), ("norm", 272, 640, 1), ("norm", 12304, 256, 1), ("plain", 272, 1152, 1),
          ("glu", 16, 128, 1), ("glu", 304, 2560, 1), ("glu", 9728, 384, 1), ("res", 48, 1536, 1),
          ("res", 2560, 4096, 1), ("parts", 2560, 4096, 2), ("parts", 2560, 9728, 4), ("parts", 1040, 512, 4)]


@pytest.mark.parametrize("kind,n,k,ksplit", SHAPES)
@pytest.mark.parametrize("rows", [9, 16, 17, 31, 33, 48, 64, 65, 100, 128])
def test_many_rows_bitexact(lib, kind, n, k, ksplit, rows):
    call = Call(lib, kind, n, k, ksplit, seed=n + k)
    x, res = rnd(rows, k, scale=2.0, seed=rows), rnd(rows, n, seed=rows + 1)
    want = [call(x[i:i + 8].contiguous(), res[i:i + 8].contiguous(), False) for i in range(0, rows, 8)]
    for wide in (True,) if rows > 64 else (True, False):
        got = call(x, res, wide)
        for j, g in enumerate(got):
            w = torch.cat([o[j] for o in want])
            assert torch.isfinite(w).all()
            kindint = torch.int16 if g.dtype == torch.bfloat16 else torch.int32
            assert torch.equal(g.contiguous().view(kindint), w.view(kindint)), (wide, j)


@pytest.mark.parametrize("kind,n,k,ksplit", [("glu", 2064, 1280, 1), ("glu", 4112, 384, 1), ("glu", 12288, 384, 1),
                                             ("parts", 4096, 1536, 4)])
@pytest.mark.parametrize("rows", [9, 24, 96, 97])
def test_units_per_workgroup_bitexact(lib, kind, n, k, ksplit, rows):
    """Widths for which the launch rule picks 2, 3, 2 or 6 or 3 (by the row
    tiles) and 4 units per workgroup, and, in qdec_gemm, k ranges short enough
    that the per-tile kernels stay."""
    test_many_rows_bitexact(lib, kind, n, k, ksplit, rows)


@pytest.mark.parametrize("rows,n,k", [(9, 16, 256), (16, 4112, 256), (33, 784, 256), (64, 16896, 256),
                                      (9, 16896, 4096), (16, 16896, 2560), (17, 16896, 2560), (24, 16896, 1024),
                                      (32, 784, 4096), (33, 16896, 2048), (48, 4112, 1152), (64, 16896, 2560)])
def test_many_rows_argmax(lib, rows, n, k):
    """The lm_head's logits and picks, grouped as the runtime groups them (two
    tiles per wave at 24 rows of k = 1024), over k ranges shorter and longer
    than the load rings; equal weight rows plant exact ties, so the lowest of
    equal indices has to win across units and workgroups."""
    from qdec.runtime import lm_tiles
    call = Call(lib, "argmax", n, k, 1, seed=n)
    w = rnd(n, k, scale=0.05, seed=n)
    w[n // 2] = w[3] = w[n - 1] = 4 * w[3]
    call.w = pack(lib, w)
    x, res = rnd(rows, k, scale=2.0, seed=rows), rnd(rows, n, seed=1)
    want = [call(x[i:i + 8].contiguous(), res[i:i + 8], False) for i in range(0, rows, 8)]
    call.tiles = lm_tiles(rows, n, k, 4, False)
    assert call.tiles == (8 if (rows, k) == (24, 1024) else 1)
    logits, ids = call(x, res, False)
    assert torch.equal(logits, torch.cat([o[0] for o in want]))
    assert torch.equal(ids, torch.cat([o[1] for o in want]))
    top = logits.float().amax(1, keepdim=True)
    first = torch.where(logits.float() == top, torch.arange(n, device=DEV), n).amin(1)
    assert torch.equal(ids, first)


@pytest.mark.parametrize("rows", [9, 40])
def test_many_rows_argmax_of_infinite_logits(lib, rows):
    """Logits of -inf, +inf and NaN: a row without a logit above -inf picks
    QDEC_NAN_ID and one of +inf its first, as the calls of up to 8 rows."""
    from qdec import capi
    n, k = 784, 1024
    call = Call(lib, "argmax", n, k, 1, seed=n)
    w = rnd(n, k, scale=0.05, seed=n)
    w[:, 0] = float("-inf")
    call.w, call.norm_w[0] = pack(lib, w), 1
    x, res = rnd(rows, k, scale=2.0, seed=rows), rnd(rows, n, seed=1)
    x[:, 0] = torch.tensor([1.0, -1.0, 0.0], device=DEV).repeat(rows)[:rows]
    x[5] = float("nan")
    logits, ids = call(x, res, False)
    want = [call(x[i:i + 8].contiguous(), res[i:i + 8], False) for i in range(0, rows, 8)]
    assert torch.equal(logits.isnan(), torch.cat([o[0] for o in want]).isnan())
    assert torch.equal(ids, torch.cat([o[1] for o in want]))
    kinds = [capi.NAN_ID if i % 3 != 1 or i == 5 else 0 for i in range(rows)]
    assert ids.tolist() == kinds
    assert (logits[0] == float("-inf")).all() and (logits[1] == float("inf")).all() and logits[2].isnan().all()


@pytest.mark.parametrize("kind,n,k,waves", [("norm", 4096, 2048, 8), ("norm", 304, 1024, 4), ("glu", 6144, 2048, 4),
                                            ("glu", 48, 1024, 4), ("res", 304, 2048, 8), ("res", 304, 9216, 4), ("plain", 304, 1024, 4),
                                            ("argmax", 304, 1024, 4), ("argmax", 4112, 2048, 8)])
def test_short_ring_bitexact(lib, kind, n, k, waves):
    """Widths whose k range per wave is a multiple of 8 but not of the longer
    load rings (rows staged in LDS, a ring of 8; without NORM_IN only a range of
    8 steps): 1, 3, 5 and 8 rows give the
    bits that a call of 12 rows, which reads them directly, gives."""
    call = Call(lib, kind, n, k, 1, seed=n + k)
    call.waves = waves
    x, res = rnd(12, k, scale=2.0, seed=5), rnd(12, n, seed=6)
    want = call(x, res, False)
    call.row_major = True
    for rows in ([3], [0, 1, 2], [7, 8, 9, 10, 11], list(range(8))):
        got = call(x[rows].contiguous(), res[rows].contiguous(), False)
        assert torch.equal(got[0].contiguous().view(torch.int16), want[0][rows].view(torch.int16)), rows
        assert all(torch.equal(g, w[rows]) for g, w in zip(got[1:], want[1:]))  # the picks


@pytest.mark.parametrize("kind,n", [("norm", 304), ("argmax", 4112)])
@pytest.mark.parametrize("rows,nparts", [(1, 2), (1, 4), (1, 5), (3, 2)])
def test_short_ring_merges_split_update(lib, kind, n, rows, nparts):
    """A pending split update merged by a call on the ring of 8: in its
    prologue at one row and up to four parts, else by the pre-pass.  The
    merged row is bf16(x + bf16(p0 + p1 + ...)), the output that of the same
    call on it."""
    k = 1024
    call = Call(lib, kind, n, k, 1, seed=n)
    x, res = rnd(rows, k, scale=2.0, seed=5), rnd(rows, n, seed=6)
    parts = torch.randn(nparts, rows, k, generator=torch.Generator().manual_seed(7)).to(DEV)
    upd = parts[0]
    for p in parts[1:]:
        upd = upd + p
    merged = (x.float() + upd.to(torch.bfloat16).float()).to(torch.bfloat16)
    want = call(merged, res, False)
    call.x_parts = parts
    got = call(x, res, False)
    assert torch.equal(call.merged.view(torch.int16), merged.view(torch.int16))
    assert all(torch.equal(g, w) for g, w in zip(got, want))


@pytest.mark.parametrize("kind,n,k", [("res", 48, 9728), ("plain", 48, 1152)])
def test_row_major_rows_bitexact(lib, kind, n, k):
    """9 to 16 row-major rows that do not fit LDS (k = 9728), or whose k range
    no load ring divides, take the direct path: the bits of fragment order."""
    call = Call(lib, kind, n, k, 1, seed=n + k)
    x, res = rnd(16, k, scale=2.0, seed=5), rnd(16, n, seed=6)
    want = call(x, res, False)[0]
    call.row_major = True
    for rows in (9, 13, 16):
        got = call(x[:rows].contiguous(), res[:rows].contiguous(), False)[0]
        assert torch.equal(got.contiguous().view(torch.int16), want[:rows].contiguous().view(torch.int16)), rows


def test_wide_refusals(lib):
    from qdec import capi
    x, out = rnd(128, 256), torch.zeros(128, 64, dtype=torch.bfloat16, device=DEV)
    good = dict(x=x.data_ptr(), w=x.data_ptr(), out=out.data_ptr(), eps=1e-6, rows=100, n=64, k=256, flags=0, ksplit=1,
                waves=4, tiles_per_wg=1, x_frag=1)
    lib.gemm_wide_workspace(capi.GemmArgs(**good))
    for bad in (dict(rows=8), dict(rows=129), dict(waves=8), dict(waves=2), dict(tiles_per_wg=2), dict(x_frag=0),
                dict(ksplit=2), dict(flags=capi.ARGMAX), dict(resident=1), dict(k=192)):
        with pytest.raises(capi.QdecError):
            lib.gemm_wide_workspace(capi.GemmArgs(**{**good, **bad}))
    with pytest.raises(capi.QdecError):  # qdec_gemm itself still ends at 64 rows
        lib.gemm_workspace(capi.GemmArgs(**good))


def test_short_prompts_of_several_lengths_in_one_state(lib):
    """One state prefills prompts of different lengths one after the other:
    each leaves what a fresh state leaves, a short one after a long one
    (unsplit products) too."""
    from qdec.checkpoint import generate_tensors, qwen3_config
    from qdec.runtime import DecodeState, DeviceModel
    cfg = qwen3_config(num_hidden_layers=2, vocab_size=1024)
    model = DeviceModel(cfg, dict(generate_tensors(cfg, seed=3, norm_jitter=0.05)), DEV)
    shared = DecodeState(model, 2, 1120, max_t=16, keep_logits=True)
    for S in (60, 25, 64, 40, 130, 33, 1100, 33, 400, 64):
        prompt = torch.randint(0, 1024, (2, S), generator=torch.Generator().manual_seed(S)).to(DEV)
        fresh = DecodeState(model, 2, 1120, max_t=16, keep_logits=True)
        for st in (shared, fresh):
            st.prefill(prompt)
        torch.cuda.synchronize()
        assert torch.equal(shared.logits[:2], fresh.logits[:2]), S
        assert torch.equal(shared.k_cache[:, :, :, :S], fresh.k_cache[:, :, :, :S]), S


@pytest.mark.parametrize("B,S,hidden", [(1, 37, 320), (3, 20, 320), (1, 64, 512), (2, 20, 512)])
def test_short_prompt_of_widths_the_wide_product_refuses(lib, monkeypatch, B, S, hidden):
    """Widths that are not all multiples of 128: a prompt of up to 64 rows is
    one pass over the weights (qdec_gemm), not one per decode step, and its
    logits, cache and picks agree with the decode steps' (bf16 sums in another
    order: 2e-2 of the largest, as every end-to-end comparison here)."""
    from qdec.checkpoint import generate_tensors, qwen3_config
    from qdec.runtime import DecodeState, DeviceModel
    cfg = qwen3_config(num_hidden_layers=2, vocab_size=1024, hidden_size=hidden, intermediate_size=704,
                       num_attention_heads=4, num_key_value_heads=2)
    model = DeviceModel(cfg, dict(generate_tensors(cfg, seed=3, norm_jitter=0.05)), DEV)
    prompt = torch.randint(0, 1024, (B, S), generator=torch.Generator().manual_seed(S)).to(DEV)
    st, ref = (DecodeState(model, B, 160, max_t=4, keep_logits=True) for _ in range(2))
    passes, embed = [], st.lib.embed
    monkeypatch.setattr(st.lib, "embed", lambda e, s: (passes.append(e.rows), embed(e, s)))
    st.prefill(prompt)
    monkeypatch.undo()
    assert passes == [B * S]
    ref.prefill_steps(prompt)
    torch.cuda.synchronize()
    t = (S - 1) % ref.max_t + 1
    logits = ref.logits[:B * t].view(B, t, -1)[:, t - 1].float()
    assert (st.logits[:B].float() - logits).abs().max() <= 2e-2 * logits.abs().max()
    for got, want in ((st.k_cache, ref.k_cache), (st.v_cache, ref.v_cache)):
        assert (got.float() - want.float()).abs().max() <= 2e-2 * want.float().abs().max()
    assert st.lens.tolist() == [S] * B


@pytest.mark.parametrize("B", [1, 2])
def test_attention_merged_in_o_on_the_short_ring(lib, monkeypatch, B):
    """16 query heads on 4 kv heads: O (k = 2048 on 8 waves, a ring of 8)
    merges the attention's chunk partials while it stages its rows; the step
    has the bits of the one whose attention merges them."""
    from qdec.checkpoint import generate_tensors, qwen3_config
    from qdec.runtime import DecodeState, DeviceModel
    cfg = qwen3_config(num_hidden_layers=2, vocab_size=1024, hidden_size=1024, intermediate_size=3072,
                       num_attention_heads=16, num_key_value_heads=4)
    model = DeviceModel(cfg, dict(generate_tensors(cfg, seed=3, norm_jitter=0.05)), DEV)
    prompt = torch.randint(0, 1024, (B, 300), generator=torch.Generator().manual_seed(B)).to(DEV)
    got = []
    for merge in (True, False):
        st = DecodeState(model, B, 640, max_t=1, keep_logits=True)
        assert st._merge_in_o(1) and st.chunk < 300
        if not merge:
            monkeypatch.setattr(st, "_merge_in_o", lambda t: False)
        st.prefill(prompt)
        for _ in range(3):
            st.run_step()
        torch.cuda.synchronize()
        got.append((st.logits[:B].clone(), st.ids[:B].clone()))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
