"""GPU parity of al_fattn_f16 against oracle O2 (the f32-accumulating
restatement of nnml_compute_forward_flash_attn_ext_f16, arm.cpp:2196-2433).

Bar: max-abs <= 2e-3 and rel-L2 <= 1e-3 on the fp32 output, identical NaN
pattern. Every case prints its name before touching the GPU.
"""
import math

import numpy as np
import pytest

from arclight_amd import abi
from oracle import oracle as O
from tests.fattn_cases import assert_parity, run_gpu

pytestmark = pytest.mark.gpu
SCALE = 1.0 / math.sqrt(128)


def _case(name):
    print(f"\n[case] {name}", flush=True)


def _check(name, q, k, v, mask=None, sinks=None, **kw):
    _case(name)
    ref = O.attention(q, k, v, mask, sinks, **kw)
    got = run_gpu(q, k, v, mask, sinks, **kw)
    assert_parity(got, ref, what=name)
    return got, ref


@pytest.mark.parametrize("explicit", [True, False])
def test_decode_qwen3_4b_c512(gpu, explicit):
    # 1 layer, q_len 1, Hq 32, Hkv 8, D 128, context 512 (+ the new token), n_kv padded to 768
    q, k, v = O.make_inputs(1234, T=1, Hq=32, Hkv=8, n_kv=768)
    if explicit:
        _check("decode c512 explicit mask", q, k, v, O.causal_mask(1, 768, 512), scale=SCALE)
    else:
        _check("decode c512 implicit", q, k, v, scale=SCALE, kv_len=513)


@pytest.mark.parametrize("ctx", [4096, 16384, 32768])
def test_decode_qwen3_4b_long(gpu, ctx):
    q, k, v = O.make_inputs(ctx, T=1, Hq=32, Hkv=8, n_kv=ctx)
    _check(f"decode ctx {ctx}", q, k, v, scale=SCALE, kv_len=ctx)


def test_decode_gqa8_qwen3_32b(gpu):
    q, k, v = O.make_inputs(7, T=1, Hq=64, Hkv=8, n_kv=4096)
    _check("decode gqa 8:1 ctx 4096", q, k, v, scale=SCALE)


@pytest.mark.parametrize("T", [2, 4, 8])
def test_verify_qwen3_8b(gpu, T):
    # speculative verify: drafts at positions C..C+T-1, causal among drafts
    C = 2048
    n_kv = 2304
    q, k, v = O.make_inputs(100 + T, T=T, Hq=32, Hkv=8, n_kv=n_kv)
    _check(f"verify T={T} explicit", q, k, v, O.causal_mask(T, n_kv, C), scale=SCALE)
    _check(f"verify T={T} implicit", q, k, v, scale=SCALE, kv_len=C + T, causal_pos0=C)


def test_verify_gqa8_t8(gpu):
    q, k, v = O.make_inputs(55, T=8, Hq=64, Hkv=8, n_kv=1024)
    _check("verify gqa8 T=8", q, k, v, scale=SCALE, kv_len=1000, causal_pos0=992)


@pytest.mark.parametrize("T,pos0", [(64, 0), (96, 160)])
def test_prefill_chunk_causal(gpu, T, pos0):
    n_kv = pos0 + T
    q, k, v = O.make_inputs(T + pos0, T=T, Hq=32, Hkv=8, n_kv=n_kv)
    _check(f"prefill T={T} pos0={pos0} explicit", q, k, v, O.causal_mask(T, n_kv, pos0), scale=SCALE)
    _check(f"prefill T={T} pos0={pos0} implicit", q, k, v, scale=SCALE, causal_pos0=pos0)


def test_streams_and_mask_broadcast(gpu):
    # two streams (nnml dim 3) with their own mask planes
    rng = np.random.default_rng(3)
    q, k, v = O.make_inputs(3, B=2, T=2, Hq=8, Hkv=2, n_kv=256)
    m = np.full((2, 1, 64, 256), -np.inf, dtype=np.float16)
    m[0, 0, :2, :100] = 0
    m[1, 0, :2, 50:230] = 0
    m[1, 0, 1, 229] = -np.inf
    _check("streams B=2", q, k, v, m, scale=SCALE)
    # per-head mask planes with finite values
    mh = rng.uniform(-3, 0, size=(1, 8, 64, 256)).astype(np.float16)
    mh[..., 200:] = -np.inf
    _check("mask per head", q, k, v, mh, scale=SCALE)


def test_sinks_softcap_alibi(gpu):
    rng = np.random.default_rng(11)
    q, k, v = O.make_inputs(11, T=3, Hq=12, Hkv=4, n_kv=320)
    sinks = rng.standard_normal(12).astype(np.float32) * 3
    m = O.causal_mask(3, 320, 300)
    _check("sinks", q, k, v, m, sinks, scale=SCALE)
    _check("softcap", q, k, v, m, scale=SCALE * 4, logit_softcap=5.0)
    alibi = m.astype(np.float32)
    alibi[0, 0, :3, :301] = -np.arange(301, dtype=np.float32)[::-1] / 64.0
    _check("alibi", q, k, v, alibi.astype(np.float16), scale=SCALE, max_bias=8.0)


def test_ragged_sizes(gpu):
    # n_kv not a multiple of 32, kv_len not a multiple of the tile, T*G = 12 rows
    q, k, v = O.make_inputs(5, T=3, Hq=8, Hkv=2, n_kv=40)
    _check("n_kv 40 kv_len 37", q, k, v, scale=SCALE, kv_len=37)
    q, k, v = O.make_inputs(6, T=5, Hq=6, Hkv=3, n_kv=33)
    _check("n_kv 33 T 5 G 2", q, k, v, O.causal_mask(5, 33, 27), scale=SCALE)


def test_all_masked_rows_are_nan_and_single_cell(gpu):
    q, k, v = O.make_inputs(9, T=2, Hq=4, Hkv=1, n_kv=64)
    m = np.full((1, 1, 64, 64), -np.inf, dtype=np.float16)
    m[0, 0, 1, 17] = 0                      # token 1 sees exactly cell 17, token 0 sees nothing
    got, ref = _check("all-masked + single cell", q, k, v, m, scale=SCALE)
    assert np.isnan(got[0, 0]).all()
    vf = v.astype(np.float32)
    np.testing.assert_allclose(got[0, 1], np.broadcast_to(vf[0, 17, 0], (4, 128)), rtol=0, atol=1e-6)


def test_garbage_in_masked_cells(gpu):
    # unwritten cache cells may hold NaN/Inf: masked cells must not leak
    q, k, v = O.make_inputs(21, T=1, Hq=32, Hkv=8, n_kv=512)
    ref = O.attention(q, k, v, scale=SCALE, kv_len=300)
    kg, vg = k.copy(), v.copy()
    kg[:, 300:] = np.float16(np.nan)
    vg[:, 300:] = np.float16(np.inf)
    _case("garbage beyond kv_len")
    got = run_gpu(q, kg, vg, scale=SCALE, kv_len=300)
    assert_parity(got, ref, what="garbage")
    m = O.causal_mask(1, 512, 299)
    _case("garbage beyond mask")
    got = run_gpu(q, kg, vg, m, scale=SCALE)
    assert_parity(got, ref, what="garbage mask")


def test_prec_default_and_determinism(gpu):
    q, k, v = O.make_inputs(31, T=1, Hq=32, Hkv=8, n_kv=2048)
    _case("determinism")
    a = run_gpu(q, k, v, scale=SCALE, prec=abi.AL_PREC_DEFAULT)
    b = run_gpu(q, k, v, scale=SCALE, prec=abi.AL_PREC_F32)
    assert np.array_equal(a, b)


def test_caller_workspace(gpu):
    from arclight_amd import device, fattn
    from arclight_amd._lib import ArclightError
    q, k, v = O.make_inputs(41, T=1, Hq=32, Hkv=8, n_kv=8192)
    ref = O.attention(q, k, v, scale=SCALE)
    dq, dk, dv = fattn.upload_q(q), fattn.upload_kv(k), fattn.upload_kv(v)
    dst = device.DeviceTensor.empty(q.shape, np.float32, axes=abi.DST_AXES)
    need = fattn.workspace_bytes(dq, dk, dv, None, None, dst, scale=SCALE)
    assert need > 0
    _case("caller workspace")
    ws = device.DeviceBuffer(need)
    ws.zero()
    for _ in range(2):
        fattn.flash_attn_ext(dq, dk, dv, scale=SCALE, dst=dst, workspace=ws)
        device.synchronize()
        assert_parity(dst.numpy(np.float32), ref, what="caller workspace")
    small = device.DeviceBuffer(need - 4)
    with pytest.raises(ArclightError) as ei:
        fattn.flash_attn_ext(dq, dk, dv, scale=SCALE, dst=dst, workspace=small)
    assert ei.value.status == abi.AL_ERR_WORKSPACE


def test_rejects_what_the_reference_asserts(gpu):
    from arclight_amd._lib import ArclightError
    q, k, v = O.make_inputs(1, T=2, Hq=8, Hkv=3 if False else 2, n_kv=64)
    short_mask = np.zeros((1, 1, 32, 64), dtype=np.float16)     # rows < PAD(T, 64)
    with pytest.raises(ArclightError) as ei:
        run_gpu(q, k, v, short_mask, scale=SCALE)
    assert ei.value.status == abi.AL_ERR_INVALID
    with pytest.raises(ArclightError) as ei:
        run_gpu(q, k, v, scale=SCALE, max_bias=1.0)              # ALiBi without mask
    assert ei.value.status == abi.AL_ERR_INVALID
    with pytest.raises(ArclightError) as ei:
        run_gpu(q, k, v, scale=SCALE, prec=3)
    assert ei.value.status == abi.AL_ERR_INVALID
    q64, k64, v64 = O.make_inputs(1, T=1, Hq=8, Hkv=2, D=64, n_kv=64)
    with pytest.raises(ArclightError) as ei:
        run_gpu(q64, k64, v64, scale=SCALE)
    assert ei.value.status == abi.AL_ERR_UNSUPPORTED


def test_split_merge_repeatable_back_to_back(gpu):
    # Multi-split calls (two merge levels) launched back to back on one stream
    # without host synchronization: every result must equal the first bit for
    # bit (the merge order is fixed) and match the oracle.
    from arclight_amd import device, fattn
    q, k, v = O.make_inputs(77, T=1, Hq=32, Hkv=8, n_kv=32768)
    ref = O.attention(q, k, v, scale=SCALE)
    dq, dk, dv = fattn.upload_q(q), fattn.upload_kv(k), fattn.upload_kv(v)
    n = 64
    dsts = [device.DeviceTensor.empty(q.shape, np.float32, axes=abi.DST_AXES) for _ in range(n)]
    _case("split merge x64 back to back")
    for rep in range(3):
        for d in dsts:
            fattn.flash_attn_ext(dq, dk, dv, scale=SCALE, dst=d)
        device.synchronize()
        outs = [d.numpy(np.float32) for d in dsts]
        if rep == 0:
            first = outs[0]
            assert_parity(first, ref, what="split merge")
        for i, o in enumerate(outs):
            assert np.array_equal(o, first), f"rep {rep} call {i} differs"


def test_shapes_alternating_on_one_workspace(gpu):
    # Calls of different shapes lay out their merge records differently; the
    # arrival counters and split flags live in a fixed region no record
    # overlaps, so alternating shapes on one workspace keeps every call
    # correct.
    from arclight_amd import device, fattn
    cases = [dict(seed=90, B=1, T=1, Hq=32, Hkv=8, n_kv=32768),
             dict(seed=91, B=2, T=2, Hq=8, Hkv=2, n_kv=2048),
             dict(seed=92, B=1, T=8, Hq=32, Hkv=8, n_kv=8192),
             dict(seed=93, B=1, T=96, Hq=32, Hkv=8, n_kv=256)]
    prepared = []
    need = 0
    for c in cases:
        seed = c.pop("seed")
        q, k, v = O.make_inputs(seed, **c)
        ref = O.attention(q, k, v, scale=SCALE)
        dq, dk, dv = fattn.upload_q(q), fattn.upload_kv(k), fattn.upload_kv(v)
        dst = device.DeviceTensor.empty(q.shape, np.float32, axes=abi.DST_AXES)
        need = max(need, fattn.workspace_bytes(dq, dk, dv, None, None, dst, scale=SCALE))
        prepared.append((dq, dk, dv, dst, ref))
    ws = device.DeviceBuffer(need)
    ws.zero()
    _case("alternating shapes, one workspace")
    for rnd in range(3):
        for order in (prepared, prepared[::-1]):
            for dq, dk, dv, dst, ref in order:
                fattn.flash_attn_ext(dq, dk, dv, scale=SCALE, dst=dst, workspace=ws)
            device.synchronize()
            for i, (dq, dk, dv, dst, ref) in enumerate(order):
                assert_parity(dst.numpy(np.float32), ref, what=f"round {rnd} call {i}")
    # the lower half of the 256 KiB counter region holds the arrival counters
    # (the upper half the decode split flags, which carry epochs)
    cnt = np.empty(32768, dtype=np.uint32)
    ws.download(cnt)
    assert not cnt.any(), "arrival counters not left at zero"


@pytest.mark.parametrize("pos0", [0, 512, 1024, 1536])
def test_prefill_kernel_chunk512_qwen3_4b(gpu, pos0):
    # each 512-token chunk of a 2048-token causal prefill (Hq 32, Hkv 8), the
    # whole output against the oracle
    n_kv = 2048
    q, k, v = O.make_inputs(500 + pos0, T=512, Hq=32, Hkv=8, n_kv=n_kv)
    _check(f"prefill chunk 512 pos0 {pos0}", q, k, v, scale=SCALE, kv_len=pos0 + 512, causal_pos0=pos0)


def test_prefill_row_tiles_by_context_and_scratch(gpu):
    """A 512-token chunk over a long context runs 128-row tiles in two
    workgroups each; with less scratch at hand (but what a shared tile of
    such a call ever needed) it runs unshared tiles, and takes 64-row tiles
    over a short one. Causal and with a mask tensor, against the oracle."""
    from arclight_amd import device, fattn
    n_kv = 7168
    q, k, v = O.make_inputs(530, T=512, Hq=32, Hkv=8, n_kv=n_kv)
    dq, dk, dv = fattn.upload_q(q), fattn.upload_kv(k), fattn.upload_kv(v)
    dst = device.DeviceTensor.empty(q.shape, np.float32, axes=abi.DST_AXES)
    ref = O.attention(q, k, v, scale=SCALE, kv_len=n_kv, causal_pos0=n_kv - 512)
    need = fattn.workspace_bytes(dq, dk, dv, None, None, dst, scale=SCALE, kv_len=n_kv, causal_pos0=n_kv - 512)
    assert need >= 128 * 2 * 128 * 528                     # records of 128 rows, two workgroups to each of 128 tiles
    assert fattn.workspace_bytes(dq, dk, dv, None, None, dst, scale=SCALE, kv_len=1024, causal_pos0=512) == 0
    for nbytes in (need, need - 4, 1 << 20):
        _case(f"prefill 512 tokens over {n_kv} cells, {nbytes} bytes of scratch")
        ws = device.DeviceBuffer(nbytes)
        ws.zero()
        fattn.flash_attn_ext(dq, dk, dv, scale=SCALE, kv_len=n_kv, causal_pos0=n_kv - 512, dst=dst, workspace=ws)
        device.synchronize()
        assert_parity(dst.numpy(np.float32), ref, what=f"{nbytes} bytes of scratch")
    m = O.causal_mask(512, n_kv, n_kv - 600, kv_len=n_kv - 88)
    _check("prefill 512 tokens, long mask tensor", q, k, v, m, scale=SCALE)


@pytest.mark.parametrize("T,Hq,Hkv,n_kv,pos0", [(33, 1, 1, 40, 0), (9, 32, 8, 17, 8), (16, 32, 8, 4096, 4000),
                                                (17, 32, 8, 3000, 2983), (63, 32, 8, 500, 437), (31, 64, 8, 2048, 1900),
                                                (51, 10, 2, 700, 100)])
def test_few_rows_on_the_prefill_kernel(gpu, T, Hq, Hkv, n_kv, pos0):
    """33 to 255 query rows per kv head without a mask tensor: one row, one
    tile and one cell either side of its 64-row tiles, causal and not, with
    sinks and softcap, and in two streams."""
    q, k, v = O.make_inputs(7000 + T, B=2 if Hkv == 2 else 1, T=T, Hq=Hq, Hkv=Hkv, n_kv=n_kv)
    name = f"{T} tokens of {Hq} heads over {n_kv} cells"
    _check(f"{name}, causal from {pos0}", q, k, v, scale=SCALE, kv_len=min(n_kv, pos0 + T), causal_pos0=pos0)
    sinks = np.random.default_rng(T).standard_normal(Hq).astype(np.float32)
    _check(f"{name}, sinks + softcap", q, k, v, None, sinks, scale=SCALE * 3, logit_softcap=4.0, kv_len=n_kv - 1)


def test_prefill_kernel_gqa8_noncausal_sinks_softcap(gpu):
    rng = np.random.default_rng(8)
    q, k, v = O.make_inputs(600, T=256, Hq=64, Hkv=8, n_kv=1000)
    _check("prefill gqa8 chunk 256 causal", q, k, v, scale=SCALE, kv_len=1000, causal_pos0=700)
    _check("prefill gqa8 non-causal kv_len 777", q, k, v, scale=SCALE, kv_len=777)
    sinks = rng.standard_normal(64).astype(np.float32)
    _check("prefill gqa8 sinks + softcap", q, k, v, None, sinks, scale=SCALE * 3, logit_softcap=4.0,
           kv_len=1000, causal_pos0=744)


def test_prefill_kernel_explicit_masks(gpu):
    # The prefill kernel reads an explicit mask itself: prefix masks (runs
    # of zeros then -inf) as per-row extents, any other mask value by value
    # in the tiles of its rows (general mode), with ALiBi, softcap, sinks,
    # per-head mask slices and two streams.
    rng = np.random.default_rng(21)
    T, n_kv = 512, 1536
    q, k, v = O.make_inputs(2101, T=T, Hq=32, Hkv=8, n_kv=n_kv)
    m = O.causal_mask(T, n_kv, 1024, kv_len=1500)
    _check("prefill, causal prefix mask", q, k, v, m, scale=SCALE)
    mb = m.copy()
    mb[0, 0, :T, :1024] = np.where(mb[0, 0, :T, :1024] == 0, rng.uniform(-3, 0, (T, 1024)), -np.inf).astype(np.float16)
    mb[0, 0, 5:40, 100:300] = -np.inf                                 # holes inside some rows
    _check("prefill, general mask with biases and holes, ALiBi", q, k, v, mb, scale=SCALE, max_bias=8.0)
    sinks = rng.standard_normal(32).astype(np.float32)
    _check("prefill, general mask, softcap + sinks", q, k, v, mb, sinks, scale=SCALE * 4, logit_softcap=5.0)
    # one mask slice per head (mask dim 2 = Hq) and two streams (dim 3 = 2)
    q2, k2, v2 = O.make_inputs(2102, B=2, T=256, Hq=16, Hkv=4, n_kv=1024)
    mh = np.broadcast_to(O.causal_mask(256, 1024, 700, kv_len=956), (2, 16, 256, 1024)).copy()
    mh[1, 3, :, 200:220] = np.float16(-2.0)
    _check("prefill, per-head general mask, 2 streams", q2, k2, v2, mh, scale=SCALE, max_bias=4.0)


def test_prefill_kernel_explicit_masks_ragged_tiles(gpu):
    # rows per kv head not a multiple of the row tile (T=510 with G=4: 2040
    # rows; T=300 with G=8: 2400 rows), so the last tile has padding rows, with
    # a prefix mask (extents) and a mask with holes (the general mode, whose
    # padding rows must read no mask values)
    for seed, T, Hq, n_kv, pos0 in ((2111, 510, 32, 1536, 1000), (2112, 300, 64, 1024, 700)):
        q, k, v = O.make_inputs(seed, T=T, Hq=Hq, Hkv=8, n_kv=n_kv)
        m = O.causal_mask(T, n_kv, pos0, kv_len=pos0 + T)
        _check(f"prefill T={T} G={Hq // 8}, ragged last tile, prefix mask", q, k, v, m, scale=SCALE)
        mh = m.copy()
        mh[0, 0, 7:T - 3, 50:90] = -np.inf                                # holes: the general mode
        mh[0, 0, T - 1, 3] = np.float16(-1.5)
        _check(f"prefill T={T} G={Hq // 8}, ragged last tile, mask with holes", q, k, v, mh, scale=SCALE)


def test_prefill_kernel_scores_outgrow_the_reference(gpu):
    # Scores that climb by several times the lazy-rescale threshold (8
    # natural units) from tile to tile for some rows, so the reference max
    # moves inside the loop, with the scores of the next tile already
    # computed against the old one; other rows fall, keeping the first
    # tile's. Dimension 0 carries the ramp: s += a * 0.25 c (cell c), a per
    # row in {-3, -1, 0, 2, 4, 6}: 1.4 a natural units per 64-cell tile.
    rng = np.random.default_rng(2201)
    for seed, T, Hq, n_kv, pos0 in ((2202, 256, 32, 1024, 768), (2203, 512, 64, 1536, 1024)):
        q, k, v = O.make_inputs(seed, T=T, Hq=Hq, Hkv=8, n_kv=n_kv)
        q[..., 0] = rng.choice(np.array([-3.0, -1.0, 0.0, 2.0, 4.0, 6.0], dtype=np.float32), size=q.shape[:-1])
        k[..., 0] = (0.25 * np.arange(n_kv)).astype(np.float16)[None, :, None]
        name = f"prefill T={T} Hq={Hq}, growing scores"
        _check(f"{name}, length / causal rule", q, k, v, scale=SCALE, kv_len=pos0 + T, causal_pos0=pos0)
        m = O.causal_mask(T, n_kv, pos0, kv_len=pos0 + T)
        _check(f"{name}, prefix mask", q, k, v, m, scale=SCALE)
        mh = m.copy()
        mh[0, 0, 3:T - 5, 40:70] = -np.inf                                # holes: the general mode
        _check(f"{name}, mask with holes", q, k, v, mh, scale=SCALE)


def test_prefill_kernel_streams_ragged(gpu):
    # two streams, rows not a multiple of 64, cells not a multiple of 32
    q, k, v = O.make_inputs(601, B=2, T=510, Hq=16, Hkv=4, n_kv=1111)
    _check("prefill B=2 T=510 ragged", q, k, v, scale=SCALE, kv_len=1100, causal_pos0=590)


def test_decode_kernel_shapes(gpu):
    # whole-cell staged decode kernel: head groups of 4, 2 and 1, two merge
    # levels with an explicit mask over two streams, exactly 16 rows per head
    q, k, v = O.make_inputs(41, B=2, T=1, Hq=32, Hkv=8, n_kv=8192)
    m = np.full((2, 1, 64, 8192), -np.inf, dtype=np.float16)
    m[0, 0, 0, :8000] = 0
    m[1, 0, 0, :6000] = 0
    m[1, 0, 0, 3000:3100] = -np.inf
    _check("decode two streams, mask, two-level merge", q, k, v, m, scale=SCALE)
    q, k, v = O.make_inputs(42, T=1, Hq=24, Hkv=6, n_kv=3000)
    _check("decode Hkv 6 (head pairs)", q, k, v, scale=SCALE, kv_len=2999)
    q, k, v = O.make_inputs(43, T=1, Hq=16, Hkv=1, n_kv=5000)
    _check("decode 16 rows on one kv head", q, k, v, scale=SCALE, kv_len=4990)
    q, k, v = O.make_inputs(44, T=2, Hq=64, Hkv=8, n_kv=1024)
    _check("verify T=2 gqa 8:1 (16 rows)", q, k, v, scale=SCALE, kv_len=1000, causal_pos0=998)


def test_decode_kernel_two_row_blocks(gpu):
    # 17..32 query rows per kv head with implicit masks: the decode kernel's
    # two-row-block form (8-draft verify), with sinks, softcap, two streams,
    # ragged row counts and a kv_len inside the last stage
    rng = np.random.default_rng(61)
    q, k, v = O.make_inputs(61, T=8, Hq=32, Hkv=8, n_kv=2304)
    sinks = rng.standard_normal(32).astype(np.float32) * 3
    _check("two row blocks, sinks", q, k, v, None, sinks, scale=SCALE, kv_len=2056, causal_pos0=2048)
    _check("two row blocks, softcap", q, k, v, scale=SCALE * 4, logit_softcap=5.0, kv_len=2056, causal_pos0=2048)
    q, k, v = O.make_inputs(62, B=2, T=5, Hq=16, Hkv=4, n_kv=1500)
    _check("two row blocks, 2 streams, 20 rows", q, k, v, scale=SCALE, kv_len=1493, causal_pos0=1488)
    q, k, v = O.make_inputs(63, T=3, Hq=56, Hkv=7, n_kv=700)
    _check("two row blocks, 24 rows, G 8", q, k, v, scale=SCALE, kv_len=650)


def test_decode_kernel_two_row_blocks_explicit_mask(gpu):
    # 17..32 rows per kv head with the f16 mask tensor: the masked
    # two-row-block decode kernel, with the causal mask of 8 drafts, a mask
    # broadcast over two streams with ALiBi biases in it, and mask stages
    # that are all zero next to ones that are not
    q, k, v = O.make_inputs(64, T=8, Hq=32, Hkv=8, n_kv=2304)
    _check("two row blocks, explicit causal mask", q, k, v, O.causal_mask(8, 2304, 2048, kv_len=2056), scale=SCALE)
    rng = np.random.default_rng(65)
    q, k, v = O.make_inputs(65, B=2, T=6, Hq=16, Hkv=4, n_kv=1024)
    m = O.causal_mask(6, 1024, 1000, kv_len=1006)
    m[..., 200:260] = rng.uniform(-3, 0, (1, 1, m.shape[2], 60)).astype(np.float16)
    m[..., 300] = -np.inf
    _check("two row blocks, mask with biases, ALiBi, 2 streams", q, k, v, m, scale=SCALE, max_bias=8.0)


def test_decode_mask_preloaded_and_per_stage(gpu, monkeypatch):
    """A decode call with a mask tensor loads each wave's mask values into LDS
    once, before its first stage, when the workgroup's share fits
    (AL_DECODE_MASK_PRE=0: with every stage instead). Both forms apply the
    same mask values in the same order, so they give the same bits, and both
    match the oracle: one token over a mask with holes and finite values
    shared by the heads, eight drafts with the causal mask among them
    (32 rows, two row blocks), four drafts with per-head mask planes, and a
    one-token call whose share is too large to preload (131072 cells, two
    mask planes that the heads alternate between: both settings take the
    per-stage form there)."""
    rng = np.random.default_rng(77)
    cases = []
    q, k, v = O.make_inputs(771, T=1, Hq=32, Hkv=8, n_kv=4096)
    m = np.zeros((1, 1, 64, 4096), np.float16)
    m[0, 0, 0, rng.choice(4096, 700, replace=False)] = -np.inf
    m[0, 0, 0, :512] = rng.uniform(-2, 0, 512).astype(np.float16)
    m[0, 0, 0, 4000:] = -np.inf
    cases.append(("one token, holes and finite values", q, k, v, m))
    q, k, v = O.make_inputs(772, T=8, Hq=32, Hkv=8, n_kv=8448)
    cases.append(("eight drafts, causal", q, k, v, O.causal_mask(8, 8448, 8192, kv_len=8200)))
    q, k, v = O.make_inputs(773, T=4, Hq=32, Hkv=8, n_kv=2048)
    mh = rng.uniform(-1, 0, size=(1, 32, 64, 2048)).astype(np.float16)
    mh[..., 1900:] = -np.inf
    mh[0, 5, 2, :1000] = -np.inf
    cases.append(("four drafts, per-head planes", q, k, v, mh))
    q, k, v = O.make_inputs(774, T=1, Hq=8, Hkv=2, n_kv=131072)
    mb = np.zeros((1, 2, 64, 131072), np.float16)
    mb[0, 0, 0, 120000:] = -np.inf
    mb[0, 1, 0, :70000] = -np.inf
    cases.append(("one token, two mask planes, 131072 cells", q, k, v, mb))
    for name, q, k, v, m in cases:
        ref = O.attention(q, k, v, m, scale=SCALE)
        _case(f"{name}: preloaded")
        monkeypatch.delenv("AL_DECODE_MASK_PRE", raising=False)
        a = run_gpu(q, k, v, m, scale=SCALE)
        _case(f"{name}: per stage")
        monkeypatch.setenv("AL_DECODE_MASK_PRE", "0")
        b = run_gpu(q, k, v, m, scale=SCALE)
        monkeypatch.delenv("AL_DECODE_MASK_PRE", raising=False)
        assert np.array_equal(a, b, equal_nan=True), f"{name}: preloaded and per-stage masks differ"
        assert_parity(a, ref, what=name)


def test_decode_two_waves_one_pass_and_tree_merge(gpu, monkeypatch):
    """The 2-wave decode shape merges its two waves' states in one pass with
    all threads when a split covers at most AL_DECODE_ONE_PASS_CELLS cells
    (512 by default), else wave 0 folds in wave 1's state (the tree). Each
    form against the oracle, and the two against each other (the same two
    weighted terms, summed in another order: within a few ulp): one token
    over 4096 and 16384 cells (128 and 512 cells per split), the Qwen3-32B
    shape (8 rows per kv head), 2-draft verify with the causal mask among
    the drafts, 2 streams, an explicit mask with holes (preloaded and per
    stage), and one split over 40 and 10 cells (the pass writes the output
    rows; a wave with one stage or none)."""
    rng = np.random.default_rng(91)
    cases = []
    for seed, n_kv in ((911, 4096), (912, 16384)):
        q, k, v = O.make_inputs(seed, T=1, Hq=32, Hkv=8, n_kv=n_kv)
        cases.append((f"one token over {n_kv} cells", q, k, v, None, dict(kv_len=n_kv)))
    q, k, v = O.make_inputs(913, T=1, Hq=64, Hkv=8, n_kv=4096)
    cases.append(("Qwen3-32B shape, 4096 cells", q, k, v, None, dict(kv_len=4096)))
    q, k, v = O.make_inputs(914, T=2, Hq=32, Hkv=8, n_kv=8192)
    cases.append(("2 drafts over 8192 cells", q, k, v, None, dict(kv_len=8192, causal_pos0=8190)))
    q, k, v = O.make_inputs(915, B=2, T=1, Hq=32, Hkv=8, n_kv=3000)
    cases.append(("2 streams, 3000 cells", q, k, v, None, dict(kv_len=3000)))
    q, k, v = O.make_inputs(916, T=1, Hq=32, Hkv=8, n_kv=6000)
    m = np.zeros((1, 1, 64, 6000), np.float16)
    m[0, 0, 0, rng.choice(6000, 900, replace=False)] = -np.inf
    m[0, 0, 0, :300] = rng.uniform(-2, 0, 300).astype(np.float16)
    cases.append(("explicit mask with holes, 6000 cells", q, k, v, m, {}))
    for seed, n_kv in ((917, 40), (918, 10)):
        q, k, v = O.make_inputs(seed, T=1, Hq=32, Hkv=8, n_kv=n_kv)
        cases.append((f"one split over {n_kv} cells", q, k, v, None, dict(kv_len=n_kv)))
    for name, q, k, v, m, kw in cases:
        ref = O.attention(q, k, v, m, scale=SCALE, **kw)
        forms = {}
        for label, cells, pre in (("one pass", None, None), ("tree", "0", None), ("one pass, mask per stage", None, "0")):
            if pre is not None and m is None:
                continue
            _case(f"{name}: {label}")
            for var, val in (("AL_DECODE_ONE_PASS_CELLS", cells), ("AL_DECODE_MASK_PRE", pre)):
                if val is None:
                    monkeypatch.delenv(var, raising=False)
                else:
                    monkeypatch.setenv(var, val)
            forms[label] = run_gpu(q, k, v, m, scale=SCALE, **kw)
            assert_parity(forms[label], ref, what=f"{name}: {label}")
        monkeypatch.delenv("AL_DECODE_ONE_PASS_CELLS", raising=False)
        monkeypatch.delenv("AL_DECODE_MASK_PRE", raising=False)
        a, b = forms["one pass"], forms["tree"]
        assert np.array_equal(np.isnan(a), np.isnan(b)), f"{name}: forms differ in NaN rows"
        np.testing.assert_allclose(a, b, rtol=2e-6, atol=1e-6, err_msg=f"{name}: one pass against tree")
        if "one pass, mask per stage" in forms:
            assert np.array_equal(a, forms["one pass, mask per stage"], equal_nan=True), f"{name}: mask forms differ"


def test_decode_two_waves_sinks_softcap_alibi_both_merges(gpu, monkeypatch):
    """One token per stream (the 2-wave shape) with attention sinks, logit
    softcap and ALiBi over a mask with finite biases, against the oracle,
    with the one-pass and the tree merge of the waves: 4096 cells (128 per
    split: one pass by default) and 20000 cells (640 per split: the tree),
    each also with the other form forced."""
    rng = np.random.default_rng(93)
    for seed, n_kv in ((931, 4096), (932, 20000)):
        q, k, v = O.make_inputs(seed, T=1, Hq=32, Hkv=8, n_kv=n_kv)
        sinks = rng.standard_normal(32).astype(np.float32) * 3
        m = np.zeros((1, 1, 64, n_kv), np.float16)
        m[0, 0, 0, :] = (-np.arange(n_kv, dtype=np.float32)[::-1] / 4096.0).astype(np.float16)
        m[0, 0, 0, rng.choice(n_kv, n_kv // 10, replace=False)] = -np.inf
        for cells in (None, "0", "100000"):
            label = {None: "default", "0": "tree", "100000": "one pass"}[cells]
            if cells is None:
                monkeypatch.delenv("AL_DECODE_ONE_PASS_CELLS", raising=False)
            else:
                monkeypatch.setenv("AL_DECODE_ONE_PASS_CELLS", cells)
            _case(f"{n_kv} cells, sinks: {label}")
            _check(f"{n_kv} cells, sinks ({label})", q, k, v, m, sinks, scale=SCALE)
            _case(f"{n_kv} cells, softcap + ALiBi: {label}")
            _check(f"{n_kv} cells, softcap + ALiBi ({label})", q, k, v, m, scale=SCALE * 4, logit_softcap=5.0,
                   max_bias=8.0)
        monkeypatch.delenv("AL_DECODE_ONE_PASS_CELLS", raising=False)


def test_verify_waves_without_stages_and_one_pass_merge(gpu):
    """The 8-wave decode shape (17-32 query rows per kv head) merges its
    waves in one pass from their own LDS rings. Short contexts leave some of
    the 8 waves with no stage at all (they reach the merge while the others
    still work), and with one split the pass writes the output rows itself:
    8 drafts (two row blocks) over 100, 700 and 5000 cells, 5 drafts (20
    rows, one row block partly valid) over 90 cells, with the causal mask
    among the drafts, against the oracle."""
    for seed, T, n_kv in ((881, 8, 100), (882, 8, 700), (883, 8, 5000), (884, 5, 90)):
        q, k, v = O.make_inputs(seed, T=T, Hq=32, Hkv=8, n_kv=n_kv)
        kw = dict(kv_len=n_kv, causal_pos0=n_kv - T)
        _case(f"{T} drafts over {n_kv} cells")
        got = run_gpu(q, k, v, scale=SCALE, **kw)
        assert_parity(got, O.attention(q, k, v, scale=SCALE, **kw), what=f"{T} drafts over {n_kv} cells")


def _sequence_mask(rng, T, n_kv, rows):
    """Token t sees a range of cells of its own (token 2 none), as a cache
    shared by several sequences gives; the cells nobody sees."""
    m = np.full((1, 1, rows, n_kv), -np.inf, dtype=np.float16)
    cuts = np.sort(rng.choice(np.arange(1, n_kv), T, replace=False))
    for t in range(T):
        if t != 2:
            m[0, 0, t, (cuts[t - 1] + 3 if t else 0):cuts[t]] = 0
    return m, np.all(m[0, 0, :T] == -np.inf, axis=0)


@pytest.mark.parametrize("B,T,n_kv", [(64, 1, 4608), (33, 1, 200), (12, 3, 2100), (16, 1, 64)])
def test_decode_leaves_out_stages_nobody_sees(gpu, B, T, n_kv):
    """Masked decode of several streams over one K/V view: each wave takes
    the 16-cell stages that some row sees, of up to 144 of its own (three
    words of results). Runs that begin and end inside a stage, the first, the
    last or no cell at all, alternate stages, finite biases, and not-a-numbers
    in the cells that no stream sees; then ALiBi, which takes every stage."""
    rng = np.random.default_rng(B * 1000 + n_kv)
    q, k, v = O.make_inputs(88 + B, B=B, T=T, Hq=32, Hkv=8, n_kv=n_kv)
    k, v = k[:1].copy(), v[:1].copy()
    m = np.full((B, 1, 64, n_kv), -np.inf, np.float16)
    for b in range(B):
        for t in range(T):
            lo, hi = sorted(rng.integers(0, n_kv, 2))
            m[b, 0, t, lo:hi + 1] = 0.0
    m[0, 0, :T] = -np.inf
    m[1, 0, :T], m[1, 0, :T, 0] = -np.inf, 0.0
    m[2, 0, :T], m[2, 0, :T, -1] = -np.inf, 0.0
    m[3, 0, 0] = np.where(np.arange(n_kv) // 16 % 2 == 1, 0.0, -np.inf)
    m[4, 0, 0] = np.where(np.arange(n_kv) % 1040 == 17, rng.uniform(-2, 0, n_kv), -np.inf)
    m[..., 16:48] = -np.inf
    assert_parity(run_gpu(q, k, v, m, scale=SCALE, max_bias=8.0),
                  O.attention(q, k, v, m, scale=SCALE, max_bias=8.0), what="ALiBi")
    dead = np.isneginf(m[:, 0, :T]).all(axis=(0, 1))
    k[:, dead], v[:, dead] = np.nan, np.nan
    _check(f"{B} streams of {T} tokens over {n_kv} cells", q, k, v, m, scale=SCALE)


@pytest.mark.parametrize("T,Hq,Hkv,n_kv", [(16, 32, 8, 4096), (9, 32, 8, 128), (17, 4, 1, 1000), (24, 32, 8, 9000),
                                           (31, 64, 8, 2048), (40, 8, 8, 520)])
def test_few_rows_with_masks(gpu, T, Hq, Hkv, n_kv):
    """33 to 255 query rows per kv head with a mask tensor, a row tile shared
    by up to 32 workgroups, each looking at the mask of its own cells:
    sequences of one cache, with not-a-numbers in the cells that nobody sees
    and a token that sees nothing; a causal prefix, which some workgroups
    take by its extent while the one with a hole takes it by value; biases
    with ALiBi; softcap and sinks; and a mask whose rows end inside their
    last 16 bytes."""
    from arclight_amd import device, fattn
    rng = np.random.default_rng(T * 100 + n_kv)
    q, k, v = O.make_inputs(9000 + T, T=T, Hq=Hq, Hkv=Hkv, n_kv=n_kv)
    rows = (T + 63) // 64 * 64
    name = f"{T} tokens of {Hq} heads over {n_kv} cells"
    m, dead = _sequence_mask(rng, T, n_kv, rows)
    kd, vd = k.copy(), v.copy()
    kd[:, dead], vd[:, dead] = np.nan, np.nan
    _check(f"{name}, sequences", q, kd, vd, m, scale=SCALE)
    m = O.causal_mask(T, n_kv, n_kv - T - 7, kv_len=n_kv - 3)
    _check(f"{name}, causal prefix", q, k, v, m, scale=SCALE)
    q2, k2 = q.copy(), k.copy()
    q2[..., 0] = rng.choice(np.array([-3.0, 0.0, 2.0, 6.0], dtype=np.float32), size=q.shape[:-1])
    k2[..., 0] = (0.1 * np.arange(n_kv) % 40).astype(np.float16)[None, :, None]
    mh = m.copy()
    mh[0, 0, 3:, n_kv // 2:n_kv // 2 + 2] = -np.inf
    _check(f"{name}, prefix with a hole, growing scores", q2, k2, v, mh, scale=SCALE)
    mb = m.copy()
    mb[0, 0, :T] = np.where(m[0, 0, :T] == 0, rng.uniform(-3, 0, (T, n_kv)), -np.inf).astype(np.float16)
    _check(f"{name}, biases, ALiBi", q, k, v, mb, scale=SCALE, max_bias=8.0)
    sinks = rng.standard_normal(Hq).astype(np.float32)
    _check(f"{name}, biases, softcap + sinks", q, k, v, mb, sinks, scale=SCALE * 3, logit_softcap=4.0)
    if n_kv == 1000:
        n = n_kv - 3
        _case(f"{name}, {n} mask columns")
        dm = device.DeviceTensor(fattn.upload_mask(mb).buf, abi.AL_TYPE_F16, (1, 1, rows, n),
                                 (rows * 2 * n_kv, rows * 2 * n_kv, 2 * n_kv, 2), 0, abi.MASK_AXES)
        out = fattn.flash_attn_ext(fattn.upload_q(q), fattn.upload_kv(np.ascontiguousarray(k[:, :n])),
                                   fattn.upload_kv(np.ascontiguousarray(v[:, :n])), dm, None, scale=SCALE)
        device.synchronize()
        ref = O.attention(q, np.ascontiguousarray(k[:, :n]), np.ascontiguousarray(v[:, :n]),
                          np.ascontiguousarray(mb[..., :n]), scale=SCALE)
        assert_parity(out.numpy(np.float32), ref, what="mask row end")


@pytest.mark.parametrize("T,n_kv", [(9, 500), (37, 2048), (64, 2048), (130, 1000)])
@pytest.mark.parametrize("scale,big", [(1.0, 49152.0), (3.0, 24576.0), (8e-6, 0.0)])
def test_query_rows_that_scaling_would_move_out_of_f16(gpu, T, n_kv, scale, big):
    """Queries that f16 holds, with a scale that would take them out of its
    range if it went into the rows before their rounding: 33 to 255 rows per
    kv head without a mask, with a prefix mask and with one that has a hole,
    and from 256 rows on masks with a hole in every row, whose row tiles are
    shared by several workgroups. Dim 0 carries the large values, exact in
    f16, against K values that keep the scores within the softmax's reach;
    with the small scale every K value is large, and scaled rows would keep
    some 7 bits."""
    q, k, v = O.make_inputs(61 + T, T=T, Hq=32, Hkv=8, n_kv=n_kv)
    rng = np.random.default_rng(T)
    if big:
        q /= 8 * scale
        q[..., 0] = big * rng.choice([-1.0, 1.0], q.shape[:-1])
        k[..., 0] = (3.0 / (big * scale) * rng.uniform(-1, 1, k.shape[:-1])).astype(np.float16)
    else:
        k *= np.float16(1e4)
    name = f"{T} tokens over {n_kv} cells, scale {scale}, |q| to {big}"
    few = T * 4 < 256
    if few:
        _check(f"{name}, causal", q, k, v, scale=scale, kv_len=n_kv, causal_pos0=n_kv - T)
    m = O.causal_mask(T, n_kv, n_kv - T, kv_len=n_kv)
    if few:
        _check(f"{name}, prefix mask", q, k, v, m, scale=scale)
    m[..., 70] = -np.inf
    _check(f"{name}, mask with a hole", q, k, v, m, scale=scale)
    m[..., 90:400] = np.where(m[..., 90:400] == 0, np.float16(-1.25), m[..., 90:400])
    _check(f"{name}, biases", q, k, v, m, scale=scale)


def test_few_rows_probabilities_follow_the_maximum(gpu):
    """63 tokens over 8192 cells (252 query rows per kv head): probabilities
    are rounded to f16 against the largest score, not against an earlier one
    that the later exceed by up to 8. Queries, keys and their product with
    the scale's share of a row are exact in 16 bits, so what is left against
    64 bits is that rounding: at most what numpy makes of it with one maximum
    for all of a row's cells (the kernel has one for each wave's share of
    them), which against the first cells' maximum would be half as much
    again."""
    T, n_kv = 63, 8192
    scale = float(np.float32(0.125) / np.float32(1.44269504))
    q, k, v = O.make_inputs(404, T=T, Hq=32, Hkv=8, n_kv=n_kv)
    q = (q * 2).astype(np.float16).astype(np.float32)
    k = (k * np.float16(1.5)).astype(np.float16)
    _case(f"{T} tokens over {n_kv} cells against 64 bits")
    got = run_gpu(q, k, v, scale=scale)
    off, most = [], []
    for h in range(0, 32, 4):
        s = q[0, :, h].astype(np.float64) @ k[0, :, h // 4].astype(np.float64).T * scale
        p, vh = np.exp(s - s.max(-1, keepdims=True)), v[0, :, h // 4].astype(np.float64)
        pr = p.astype(np.float16).astype(np.float64)
        exact = p @ vh / p.sum(-1, keepdims=True)
        off.append(np.linalg.norm(got[0, :, h] - exact))
        most.append(np.linalg.norm(pr @ vh / pr.sum(-1, keepdims=True) - exact))
    assert np.linalg.norm(off) <= np.linalg.norm(most), (np.linalg.norm(off), np.linalg.norm(most))


@pytest.mark.parametrize("T,Hq,n_kv", [(10, 32, 700), (25, 64, 1500), (150, 32, 300)])
def test_negative_scale(gpu, T, Hq, n_kv):
    """Scores times a negative scale, without a mask and with one: calls of
    more than 32 rows per kv head stay on the split-KV kernel (its 64-row
    tiles), one workgroup to a tile and several."""
    q, k, v = O.make_inputs(71 + T, T=T, Hq=Hq, Hkv=8, n_kv=n_kv)
    _check(f"{T} tokens of {Hq} heads, scale < 0, causal", q, k, v, scale=-SCALE, kv_len=n_kv, causal_pos0=n_kv - T)
    _check(f"{T} tokens of {Hq} heads, scale < 0", q, k, v, scale=-SCALE, kv_len=n_kv - 9)
    _check(f"{T} tokens of {Hq} heads, scale < 0, mask", q, k, v, O.causal_mask(T, n_kv, n_kv - T), scale=-SCALE)


@pytest.mark.parametrize("G", [1, 17])
def test_more_streams_than_the_decode_kernel_counts(gpu, G):
    """4097 streams of 8 kv heads, more (stream, head) pairs than arrival
    counters, without a mask: the split-KV kernel's 16- and 32-row tiles. A
    sample of streams against the oracle."""
    B, n_kv = 4097, 40
    rng = np.random.default_rng(G)
    q = rng.standard_normal((B, 1, 8 * G, 128), dtype=np.float32)
    _, k, v = O.make_inputs(72, T=1, Hq=8, Hkv=8, n_kv=n_kv)
    _case(f"{B} streams of {G} heads to a kv head")
    got = run_gpu(q, k, v, scale=SCALE, kv_len=n_kv - 3)
    sel = np.unique(np.concatenate([[0, 1, B - 1], rng.choice(B, 20, replace=False)]))
    assert_parity(got[sel], O.attention(np.ascontiguousarray(q[sel]), k, v, scale=SCALE, kv_len=n_kv - 3),
                  what=f"{G} heads to a kv head")


@pytest.mark.parametrize("kw", [{}, {"max_bias": 8.0}, {"logit_softcap": 20.0}])
@pytest.mark.parametrize("T,n_kv", [(9, 500), (16, 4096), (37, 3000), (256, 2048)])
def test_masks_of_the_lowest_value(gpu, T, n_kv, kw):
    """Tokens whose every cell has f16's lowest finite value for a mask: the
    result is that of the scores alone, but for the sums' last bit, 1/256
    beside 65504. The operator's definition, which the oracle restates, has
    that rounding too; the kernel's splits add no other to it (their maxima
    and weights are exact in these units): at most 1.25 of the oracle's
    distance from 64 bits over a sample of heads."""
    q, k, v = O.make_inputs(5 + T, T=T, Hq=32, Hkv=8, n_kv=n_kv)
    m = O.causal_mask(T, n_kv, n_kv - T)
    m[0, 0, 0] = -65504
    m[0, 0, 2] = -65504
    m[0, 0, 2, 100:200] = -np.inf
    _case(f"{T} tokens over {n_kv} cells, two of the lowest mask value, {kw}")
    got, ref = run_gpu(q, k, v, m, scale=SCALE, **kw), O.attention(q, k, v, m, scale=SCALE, **kw)
    rest = [t for t in range(T) if t not in (0, 2)]
    assert_parity(got[:, rest], ref[:, rest], what="the other tokens")
    off, oracle = [], []
    for t in (0, 2):
        for h in range(0, 32, 2):
            s = q[0, t, h].astype(np.float64) @ k[0, :, h // 4].astype(np.float64).T * SCALE
            if "logit_softcap" in kw:
                s = 20 * np.tanh(s / 20)
            p = np.where(np.isneginf(m[0, 0, t]), 0.0, np.exp(s - s.max()))
            exact = p @ v[0, :, h // 4].astype(np.float64) / p.sum()
            off.append(got[0, t, h] - exact)
            oracle.append(ref[0, t, h] - exact)
    assert np.linalg.norm(off) <= 1.25 * np.linalg.norm(oracle), (np.linalg.norm(off), np.linalg.norm(oracle))
