"""CPU checks of the C ABI: the library loads, exports every entry point
include/gdnx.h declares, and rejects bad arguments before touching a GPU."""
import ctypes
import os
import re

import pytest
import torch

from gdnx_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    names = []
    for f in os.listdir(os.path.join(ROOT, "include")):
        if f.endswith(".h"):
            text = open(os.path.join(ROOT, "include", f)).read()
            text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
            names += re.findall(r"\b(gdnx_[a-z0-9_]+)\s*\(", text)
    return sorted(set(names))


def test_library_exports_every_declared_symbol():
    lib = _lib.load()
    declared = _declared()
    assert len(declared) >= 6
    missing = [n for n in declared if not hasattr(lib, n)]
    assert not missing, missing
    assert set(declared) == set(_lib.SIGNATURES), "binding signatures out of sync with the header"


def test_abi_version_and_sizes():
    lib = _lib.load()
    assert lib.gdnx_abi_version() == _lib.ABI_VERSION
    assert lib.gdnx_delta_chunk_size(128, _lib.DTYPE_BF16) == 64
    assert lib.gdnx_delta_train_chunk_size(128, _lib.DTYPE_BF16) == 32
    assert lib.gdnx_delta_chunk_size(100, _lib.DTYPE_BF16) == 0
    # per-chunk form (more than 4 lanes): per chain and chunk one d x d state and
    # one C x d block of net writes, then the chunk operands (T and Aq as C x C,
    # four float32 factors per token)
    assert lib.gdnx_delta_chunk_states_bytes(1, 4096, 16, 5, 128, 32, _lib.DTYPE_BF16) == \
        16 * 5 * 128 * ((128 * 128 + 32 * 128) * 2 + 2 * 32 * 32 * 2 + 4 * 32 * 4)
    # checkpointed form (bf16, <= 4 lanes): one state per 256-token segment,
    # the net writes and operands of every chunk
    chains, nseg = 4 * 16 * 4, 16
    assert lib.gdnx_delta_chunk_states_bytes(4, 4096, 16, 4, 128, 32, _lib.DTYPE_BF16) == \
        chains * (nseg * 128 * 128 * 2 + 128 * (32 * 128 * 2 + 2 * 32 * 32 * 2 + 4 * 32 * 4))
    # 64-token chunks: the per-chunk form whatever the lane count
    nch = 64
    assert lib.gdnx_delta_chunk_states_bytes(4, 4096, 16, 4, 128, 64, _lib.DTYPE_BF16) == \
        chains * nch * ((128 * 128 + 64 * 128) * 2 + 2 * 64 * 64 * 2 + 4 * 64 * 4)
    # backward workspace, checkpointed form: the state gradient at every
    # segment end, then dB and P3 = R dS^T per token (bf16), then k.P3 per
    # token (float32), then (more than two lanes) the float32 dq / dk / dv
    # carry between lane pairs
    ckpt = chains * ((nseg * 128 * 128 + 2 * 128 * 32 * 128) * 2 + 128 * 32 * 4)
    assert lib.gdnx_delta_bwd_workspace_bytes(4, 4096, 16, 4, 128, 32, _lib.DTYPE_BF16) == \
        (ckpt + 255) // 256 * 256 + 3 * 4 * 16 * nseg * 256 * 128 * 4
    ckpt2 = 4 * 16 * 2 * ((nseg * 128 * 128 + 2 * 128 * 32 * 128) * 2 + 128 * 32 * 4)
    assert lib.gdnx_delta_bwd_workspace_bytes(4, 4096, 16, 2, 128, 32, _lib.DTYPE_BF16) == (ckpt2 + 255) // 256 * 256
    # few heads or tokens: segments of 128 or 64 tokens, the carry of as many
    for BH, T, seg in ((16, 1999, 128), (4, 1000, 64), (2, 40, 64)):
        nseg, nch = -(-T // seg), -(-T // 32)
        ckpt = BH * 4 * ((nseg * 128 * 128 + 2 * nch * 32 * 128) * 2 + nch * 32 * 4)
        assert lib.gdnx_delta_bwd_workspace_bytes(1, T, BH, 4, 128, 32, _lib.DTYPE_BF16) == \
            (ckpt + 255) // 256 * 256 + 3 * BH * nseg * seg * 128 * 4
    # more than 4 lanes: the per-chunk form with its key-half partials
    assert lib.gdnx_delta_bwd_workspace_bytes(1, 128, 1, 5, 128, 64, _lib.DTYPE_BF16) == \
        5 * 2 * (128 * 128 + 64 * 128) * 2 + 2 * 3 * 128 * 5 * 4
    assert lib.gdnx_delta_bwd_workspace_bytes(1, 100, 1, 1, 64, 48, _lib.DTYPE_F32) == -1
    assert lib.gdnx_delta_chunk_states_bytes(1, 100, 1, 1, 64, 0, _lib.DTYPE_F32) == \
        4 * ((64 * 64 + 32 * 64) * 4 + 2 * 32 * 32 * 4 + 4 * 32 * 4)
    assert lib.gdnx_delta_fwd_workspace_bytes(1, 100, 1, 1, 64, 0, _lib.DTYPE_F32) == 4 * (2 * 32 * 32 * 4 + 4 * 32 * 4)
    assert lib.gdnx_delta_chunk_states_bytes(1, 100, 1, 1, 64, 48, _lib.DTYPE_F32) == -1


def _fwd(lib, **over):
    args = dict(q=16, k=16, v=16, ae=32, aw=32, g=32, s0=None, y=64, so=None, cs=None, ws=None,
                B=1, T=8, H=1, M=1, D=64, C=0, dt=_lib.DTYPE_F32)
    args.update(over)
    vp = lambda x: None if x is None else ctypes.c_void_p(x)
    return lib.gdnx_delta_chunk_fwd(vp(args["q"]), vp(args["k"]), vp(args["v"]), vp(args["ae"]),
                                    vp(args["aw"]), vp(args["g"]), vp(args["s0"]), vp(args["y"]),
                                    vp(args["so"]), vp(args["cs"]), vp(args["ws"]), args["B"], args["T"], args["H"],
                                    args["M"], args["D"], args["C"], args["dt"], None)


@pytest.mark.parametrize("over,code,msg", [
    (dict(q=None), -1, "non-null"),
    (dict(k=24), -1, "aligned"),
    (dict(dt=7), -1, "dtype"),
    (dict(D=96), -2, "head_dim"),
    (dict(B=0), -2, "sizes"),
    (dict(C=48), -2, "chunk"),
    (dict(y=None), -1, "non-null"),
])
def test_forward_rejects_bad_arguments(over, code, msg):
    lib = _lib.load()
    rc = _fwd(lib, **over)
    assert rc == code
    assert msg in lib.gdnx_last_error().decode()


def test_backward_requires_stash_and_workspace():
    lib = _lib.load()
    vp = ctypes.c_void_p
    ptrs = [vp(16)] * 7 + [None, None, None] + [vp(16)] * 6 + [None]
    rc = lib.gdnx_delta_chunk_bwd(*ptrs, 1, 8, 1, 1, 64, 0, _lib.DTYPE_F32, None)
    assert rc == -3
    assert "workspace" in lib.gdnx_last_error().decode()


def test_prep_requires_workspace():
    lib = _lib.load()
    vp = ctypes.c_void_p
    rc = lib.gdnx_delta_chunk_prep(vp(16), vp(16), vp(16), vp(16), vp(16), None, 1, 8, 1, 1, 64, 0,
                                   _lib.DTYPE_F32, None)
    assert rc == -3
    assert "workspace" in lib.gdnx_last_error().decode()
    rc = lib.gdnx_delta_chunk_prep(vp(16), vp(16), None, vp(16), vp(16), vp(16), 1, 8, 1, 1, 64, 0,
                                   _lib.DTYPE_F32, None)
    assert rc == -1


def test_lane_sum_rejects_bad_arguments():
    """gdnx_lane_sum checks dtype, shape and pointers before any launch."""
    lib = _lib.load()
    vp = ctypes.c_void_p
    assert lib.gdnx_lane_sum(vp(16), vp(16), 4, 4, 128, _lib.DTYPE_F64, None) == -1   # GDNX_ERR_ARG
    assert lib.gdnx_lane_sum(vp(16), vp(16), 4, 4, 100, _lib.DTYPE_F32, None) == -2   # GDNX_ERR_SHAPE
    assert lib.gdnx_lane_sum(vp(16), vp(16), 4, 0, 128, _lib.DTYPE_F32, None) == -2
    assert lib.gdnx_lane_sum(None, vp(16), 4, 4, 128, _lib.DTYPE_BF16, None) == -1
    assert lib.gdnx_lane_sum(vp(8), vp(16), 4, 4, 128, _lib.DTYPE_BF16, None) == -1     # misaligned
    assert lib.gdnx_lane_sum(None, None, 0, 4, 128, _lib.DTYPE_BF16, None) == 0          # nothing to do


@pytest.mark.parametrize("M,K", [(4, 128), (4, 64), (3, 96), (2, 8), (1, 4), (4, 256)])
def test_lane_rope_pairs_follow_the_oracle_rule(M, K):
    """The library's lane RoPE pairs (host-only call) equal the oracle's
    restatement of _lane_rope_factors; identity lanes are 0."""
    from gdnx_amd import ops
    from oracle import gdn3_layer as gl
    want = [0 if ident else d for d, _, _, ident in gl.lane_rope_params(M, K)]
    assert ops.gdn3_lane_rope_pairs(M, K) == want


def test_lane_rope_tables_match_the_oracle():
    """The product's table builder (torch float32 ops, here on the CPU) equals
    the oracle's tables bitwise."""
    from gdnx_amd import layer
    from oracle import gdn3_layer as gl
    for M, T, K in ((4, 37, 128), (4, 9, 64)):
        c1, s1 = layer.lane_rope_tables(M, T, K, "cpu")
        c2, s2 = gl.lane_rope_tables(M, T, K)
        for m, (d, _, _, ident) in enumerate(gl.lane_rope_params(M, K)):
            if ident:
                continue
            assert torch.equal(c1[m, :, :d], c2[m, :, :d]) and torch.equal(s1[m, :, :d], s2[m, :, :d])


def test_layer_boundary_entry_points_reject_bad_arguments():
    lib = _lib.load()
    vp = ctypes.c_void_p
    p16 = [vp(16)] * 15
    assert lib.gdnx_gdn3_prologue_fwd(*p16, 1, 4, 1, 5, 128, 128, 0.999, _lib.DTYPE_BF16, None) == -2
    assert "lanes" in lib.gdnx_last_error().decode()
    assert lib.gdnx_gdn3_prologue_fwd(*p16, 1, 4, 1, 4, 130, 128, 0.999, _lib.DTYPE_BF16, None) == -2
    assert "key_dim" in lib.gdnx_last_error().decode()
    bad = [vp(16)] * 2 + [vp(24)] + [vp(16)] * 12
    assert lib.gdnx_gdn3_prologue_fwd(*bad, 1, 4, 1, 4, 128, 128, 0.999, _lib.DTYPE_BF16, None) == -1
    assert lib.gdnx_gdn3_prologue_bwd(*([vp(16)] * 19 + [None]), 1, 4, 1, 4, 128, 128, 0.999,
                                      _lib.DTYPE_F32, None) == -1
    assert lib.gdnx_gdn3_epilogue_fwd(vp(16), vp(16), vp(16), vp(16), 1, 4, 1, 4, 130, 3, None) == -1
    assert "dtype" in lib.gdnx_last_error().decode()
    assert lib.gdnx_gdn3_epilogue_bwd(*([vp(16)] * 7 + [None]), 1, 4, 1, 4, 128, _lib.DTYPE_F32, None) == -1
    assert lib.gdnx_gdn3_epilogue_workspace_bytes(4, 4096, 16, 128) == 2048 * 128 * 4
    assert lib.gdnx_gdn3_epilogue_workspace_bytes(1, 3, 1, 128) == 1 * 128 * 4
    assert lib.gdnx_gdn3_epilogue_workspace_bytes(1, 17, 1, 64) == 2 * 64 * 4


def test_gdn3_compaction_count_from_a_start_position():
    lib = _lib.load()
    f = lib.gdnx_gdn3_num_compactions_from
    assert f(0, 64, 16, 16) == 4           # after tokens 15, 31, 47, 63
    assert f(5, 40, 16, 16) == 2           # tokens 5..44: after 15 and 31
    assert f(30, 2, 16, 16) == 1           # token 31 closes an interval
    assert f(37, 100, 16, 48) == 2         # after 47 and 95
    assert f(0, 0, 16, 16) == 0
    assert f(-1, 4, 16, 16) == -1 and f(0, 4, 16, 24) == -1
    assert lib.gdnx_gdn3_num_compactions(64, 16, 32) == f(0, 64, 16, 32)


def _g3_state_fwd(lib, A0=16, B0=16, U0=16, Vb0=16, t0=0, D=128, P=16, Kc=16, ws=16, mode=0):
    vp = lambda x: None if x is None else ctypes.c_void_p(x)
    return lib.gdnx_gdn3_chunk_fwd_state(vp(16), vp(16), vp(16), 1, vp(16), vp(16), 1, vp(16), vp(16),
                                         vp(A0), vp(B0), vp(U0), vp(Vb0), t0, vp(16), None, None, None, None, None,
                                         vp(ws), 1, 8, 1, 1, D, 4, P, Kc, 16 if D == 128 else 8,
                                         16 if D == 128 else 8, 8, 8, 0.97, _lib.DTYPE_F32, mode, None)


def test_gdn3_state_forward_rejects_bad_arguments():
    lib = _lib.load()
    assert _g3_state_fwd(lib, B0=None) == -1
    assert "all be given" in lib.gdnx_last_error().decode()
    assert _g3_state_fwd(lib, t0=-3) == -2
    assert "t0" in lib.gdnx_last_error().decode()
    assert _g3_state_fwd(lib, P=48, Kc=48) == -2
    assert "P=48" in lib.gdnx_last_error().decode()
    assert _g3_state_fwd(lib, P=32) == -2   # compact_every 16 is not a multiple of 32
    assert "compact_every" in lib.gdnx_last_error().decode()
    assert _g3_state_fwd(lib, Kc=24) == -2
    assert _g3_state_fwd(lib, ws=None) == -1
    assert _g3_state_fwd(lib, mode=2) == -1
    assert "compact_mode" in lib.gdnx_last_error().decode()


def _g3_decode(lib, pos=16, A=16, qkv_lanes=1, gate_ch=1, NS=2, slots=None, P=16):
    vp = lambda x: None if x is None else ctypes.c_void_p(x)
    return lib.gdnx_gdn3_decode_step(vp(16), vp(16), vp(16), qkv_lanes, vp(16), vp(16), gate_ch, vp(16), vp(16),
                                     vp(A), vp(16), vp(16), vp(16), vp(slots), vp(pos), vp(16), None, NS, 4, 2, 2,
                                     128, 4, P, 16, 16, 16, 8, 8, 0.97, _lib.DTYPE_BF16, 0, None)


def test_gdn3_decode_step_rejects_bad_arguments():
    lib = _lib.load()
    assert _g3_decode(lib, pos=None) == -1
    assert "pos" in lib.gdnx_last_error().decode()
    assert _g3_decode(lib, A=24) == -1
    assert "aligned" in lib.gdnx_last_error().decode()
    assert _g3_decode(lib, qkv_lanes=3) == -2
    assert _g3_decode(lib, gate_ch=5) == -2
    assert _g3_decode(lib, NS=0) == -2
    assert _g3_decode(lib, P=48) == -2


def test_chan_decode_step_rejects_bad_arguments():
    lib = _lib.load()
    vp = ctypes.c_void_p
    args = [vp(16)] * 7 + [None, vp(16)]
    assert lib.gdnx_delta_decode_step_chan(*args, 2, 0, 1, 1, 96, _lib.DTYPE_F32, None) == -2
    assert "head_dim" in lib.gdnx_last_error().decode()
    bad = [vp(16)] * 6 + [vp(24), None, vp(16)]
    assert lib.gdnx_delta_decode_step_chan(*bad, 2, 0, 1, 1, 128, _lib.DTYPE_F32, None) == -1
    assert lib.gdnx_delta_decode_step_chan(*([vp(16)] * 5 + [None, vp(16), None, vp(16)]), 2, 0, 1, 1, 128,
                                           _lib.DTYPE_F32, None) == -1


def test_decode_cache_host_slot_logic():
    """Slot bookkeeping runs on the host: a free list checked as a whole and
    duplicate rows refused before any launch (CPU tensors stand in for the
    pool; no compute call is made)."""
    from gdnx_amd.decode_cache import DecodeStateCache
    for kind in ("dense", "gdn3"):
        c = DecodeStateCache(4, 2, 2, 64, device="cpu", kind=kind)
        a, b, d = c.alloc(3)
        with pytest.raises(ValueError):
            c.free([a, a])
        assert len(c._free) == 1            # nothing freed by the failed call
        with pytest.raises(ValueError):
            c.free([a, 3 if 3 not in (a, b, d) else 0])
        assert len(c._free) == 1
        c.free([a, b])
        assert len(c._free) == 3
        with pytest.raises(ValueError):
            c._slot_tensor([d, -1, d])
        with pytest.raises(ValueError):       # the same check on a slot tensor
            c._slot_tensor(torch.tensor([d, -1, d], dtype=torch.int32))
        assert c._slot_tensor([d, -1, -1]).tolist() == [d, -1, -1]
    with pytest.raises(ValueError):
        DecodeStateCache(2, 2, 2, 64, device="cpu", kind="chan")
    g = DecodeStateCache(3, 2, 2, 64, device="cpu", kind="gdn3", P=32)
    s0, s1 = g.alloc(2)
    g.pos[s0] = 5
    with pytest.raises(ValueError):         # prefill of slots at different token counts
        g.prefill([s0, s1], *([torch.zeros(2, 3, 2, 64)] * 3 + [torch.zeros(2, 3, 2, 2)] * 3))


def test_gdn3_decode_step_rejects_negative_positions():
    """A negative token position has no residual slot: the host wrapper
    refuses it before any launch (the kernels treat a negative device-side
    position as an empty row)."""
    from gdnx_amd import gdn3
    NS, H, M, D = 2, 1, 1, 64
    x = torch.zeros(NS, H, D)
    gates = torch.zeros(NS, H, M)
    N = NS * H * M
    state = (torch.zeros(N, 4, 8, 8), torch.zeros(N, 4, 8, 8), torch.zeros(N, D, 16), torch.zeros(N, D, 16))
    with pytest.raises(ValueError, match="positions"):
        gdn3.gdn3_decode_step(x, x, x, gates, gates, gates, state, [3, -1], factors=(8, 8, 8, 8))


def test_noalloc_scratch_holds_what_its_query_says():
    """gdnx_gdn3_workspace_bytes > gdnx_gdn3_noalloc_scratch_bytes is the
    documented test for a call that the entry refuses.  What a workspace holds
    beside the chains' states (the runs of long intervals) must not move that
    line: it lies where the states alone (Kronecker matrix, factors, window,
    log decay, each rounded to 256 bytes) fill the scratch."""
    from gdnx_amd import _lib
    lib = _lib.load()
    cap = lib.gdnx_gdn3_noalloc_scratch_bytes()

    def up(x):
        return (x + 255) // 256 * 256
    for D in (64, 128):
        for P in (16, 32, 64):
            for dt, cb in ((_lib.DTYPE_BF16, 2), (_lib.DTYPE_F32, 4)):
                fit = 0
                for N in range(1, 6000):
                    state = (up(N * D * D * cb) + up(N * 4 * ((256 if D == 128 else 64) + 64) * 4)
                             + 2 * up(N * P * D * 4) + up(N * 4))
                    ws = lib.gdnx_gdn3_workspace_bytes(1, N, 1, D, P, dt)
                    assert ws >= state
                    assert (ws <= cap) == (state <= cap), (D, P, dt, N)
                    fit += ws <= cap
                assert 0 < fit < 5999


def test_noalloc_forward_refuses_before_any_launch():
    """The allocation-free GDN3 forward checks its static scratch's size
    before touching a device: too many chains is GDNX_ERR_WORKSPACE here too."""
    lib = _lib.load()
    assert lib.gdnx_gdn3_noalloc_scratch_bytes() == 64 << 20
    vp = ctypes.c_void_p
    rc = lib.gdnx_gdn3_chunk_fwd_state_noalloc(vp(256), vp(256), vp(256), 1, vp(256), vp(256), 1, vp(256), vp(256),
                                               None, None, None, None, 0, vp(256), None, None, None, None, None,
                                               64, 32, 16, 4, 128, 4, 16, 32, 16, 16, 8, 8, 0.97,
                                               _lib.DTYPE_BF16, 0, None)
    assert rc == -3
    assert "scratch" in lib.gdnx_last_error().decode()
    if not torch.cuda.is_available():
        # K_c = P = 16 is one fused launch with no scratch: not refused for its
        # size (with no device it then fails at its first HIP call)
        rc = lib.gdnx_gdn3_chunk_fwd_state_noalloc(vp(256), vp(256), vp(256), 1, vp(256), vp(256), 1, vp(256),
                                                   vp(256), None, None, None, None, 0, vp(256), None, None, None,
                                                   None, None, 64, 32, 16, 4, 128, 4, 16, 16, 16, 16, 8, 8, 0.97,
                                                   _lib.DTYPE_BF16, 0, None)
        assert rc == -4, lib.gdnx_last_error().decode()


def test_hip_and_nonfinite_error_codes():
    """GDNX_ERR_HIP (-4): a call that passes argument checking fails at its
    first HIP call when there is no device; the -5 code maps to
    GdnxNonFinite.  (With a GPU present the launches would run on the fake
    pointers, so the first half only runs on a machine without one.)"""
    lib = _lib.load()
    with pytest.raises(_lib.GdnxNonFinite):
        _lib.check(_lib.ERR_NONFINITE, "probe")
    for rc, cls in ((-1, _lib.GdnxError), (-2, _lib.GdnxError), (-3, _lib.GdnxError), (-4, _lib.GdnxError)):
        with pytest.raises(cls):
            _lib.check(rc, "probe")
    assert lib.gdnx_check_finite(ctypes.c_void_p(256), 8, 9, None) == -1
    assert lib.gdnx_check_finite(None, 8, _lib.DTYPE_F32, None) == -1
    assert lib.gdnx_check_finite(None, -1, _lib.DTYPE_F32, None) == -1
    prev = lib.gdnx_set_check_finite(1)
    assert lib.gdnx_set_check_finite(prev) == 1
    if torch.cuda.device_count() > 0:
        pytest.skip("a GPU is present: the no-device half of this test would launch on fake pointers")
    assert _fwd(lib) == -4
    assert lib.gdnx_last_error().decode()
    assert lib.gdnx_check_finite(ctypes.c_void_p(256), 8, _lib.DTYPE_F32, None) == -4
    assert "device" in lib.gdnx_last_error().decode()
