"""CPU-side checks of the C-ABI boundary: the shared library loads, exports every symbol the
header declares, and rejects every host-checkable bad argument with an error code before any
device work (so these run without a GPU)."""
import ctypes as C
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "spiral_mi355.h")


@pytest.fixture(scope="module")
def L():
    from ml import _lib
    return _lib


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(sp_[a-z0-9_]+)\s*\(", text)))


def test_header_symbols_exported(L):
    names = declared_functions()
    assert len(names) >= 14
    for n in names:
        assert hasattr(L.lib, n), "libspiral_mi355.so does not export %s" % n
        assert n in L.SIGNATURES, "ml/_lib.py has no ctypes signature for %s" % n


def test_missing_library_fails_loudly(L, tmp_path):
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        L.load(str(tmp_path / "libspiral_mi355.so"))


def _err(L):
    return L.lib.sp_last_error_string().decode()


def test_gemm_argument_errors(L):
    lib = L.lib
    p = C.c_void_p(0x1000)
    args = lambda **kw: [kw.get("din", 2), kw.get("dout", 0), kw.get("A", p), kw.get("B", p), kw.get("C", p),
                         kw.get("bias", None), kw.get("M", 64), kw.get("N", 64), kw.get("K", 64),
                         kw.get("alpha", 1.0), 0.0, 0, None]
    assert lib.sp_gemm_abt(*args(A=None)) == -1 and "A is NULL" in _err(L)
    assert lib.sp_gemm_abt(*args(B=C.c_void_p(0x1004))) == -3 and "16-byte" in _err(L)
    assert lib.sp_gemm_abt(*args(M=0)) == -2
    assert lib.sp_gemm_abt(*args(K=60)) == -2 and "multiple of 8" in _err(L)
    assert lib.sp_gemm_abt(*args(din=0, K=6)) == -2 and "multiple of 4" in _err(L)
    assert lib.sp_gemm_abt(*args(din=7)) == -4
    assert lib.sp_gemm_abt(*args(din=1, dout=2)) == -4
    assert lib.sp_gemm_abt(*args(alpha=0.0)) == -5 and "alpha must not be zero" in _err(L)
    # what the kernels cannot address is refused on the host: rows longer than 512 MiB (32-bit lane offsets),
    # more blocks than a launch can number
    assert lib.sp_gemm_abt(*args(K=(1 << 28) + 8)) == -2 and "too large" in _err(L)
    assert lib.sp_gemm_abt(*args(din=0, K=(1 << 27) + 4)) == -2 and "too large" in _err(L)
    assert lib.sp_gemm_abt(*args(M=1 << 20, N=1 << 20)) == -2 and "too large" in _err(L)
    assert lib.sp_gemm_abt(*args(M=(1 << 31) + 1)) == -2


@pytest.mark.parametrize("m,n,k,tile", [(11200, 1792, 32, 64), (2688, 5760, 64, 64), (2112, 1536, 96, 64), (7872, 448, 1888, 64),
                                        (10688, 768, 3648, 128), (8192, 8192, 4096, 256)])
def test_f32_tile_choice_by_the_length_of_k(L, m, n, k, tile):
    """The tile that was measured to be the fastest, where the large ones do not pay for their prologue (256 units)."""
    out = [C.c_int32() for _ in range(4)]
    assert L.lib.sp_gemm_config(0, m, n, k, *[C.byref(o) for o in out]) == 0
    assert [o.value for o in out[:2]] == [tile, tile]


def test_odd_widths_of_the_shortest_k_take_one_thread_per_output(L):
    """As far as that was measured to be faster than any tile; a batch like its members in f32."""
    out = [C.c_int32() for _ in range(5)]
    for dtype, m, n, k, each in ((2, 18043, 3, 16, True), (1, 375, 793, 16, True), (2, 20, 33, 8, True), (0, 25058, 6, 4, True), (0, 667, 134, 16, True),
                                 (0, 810, 1377, 16, False), (2, 1405, 718, 24, False), (2, 270, 47, 48, False), (2, 376, 792, 16, False)):
        for e in (1, 5):
            assert L.lib.sp_gemm_batched_config(dtype, m, n, k, e, *[C.byref(o) for o in out]) == 0
            if e == 1 or dtype == 0:
                assert (out[4].value == 0) == each and (out[0].value == 0) == each, (dtype, m, n, k, e)


def test_odd_widths_of_short_k_split_as_long_as_that_is_faster(L):
    out = [C.c_int32() for _ in range(5)]
    for m, n, k, parts in ((375, 793, 40, 4), (1745, 163, 64, 4), (1650, 1102, 192, 1), (1304, 1979, 40, 1), (376, 792, 16, 1)):
        assert L.lib.sp_gemm_batched_config(2, m, n, k, 1, *[C.byref(o) for o in out]) == 0
        assert out[4].value == parts, (m, n, k)


@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_tall_outputs_get_tiles_a_launch_can_number(L, dtype):
    """HIP launches fewer than 2^32 work items along a dimension: outputs of a few columns and up to 2^31 - 256 rows are within the
    limits of the entry point and must not be cut into tiles too small for that."""
    for m in (1 << 20, 1 << 28, (1 << 30) - 64, 1 << 30, 1200000000, (1 << 31) - 256):
        for n in (1, 4, 15, 16, 64, 128, 256):
            for k in (8, 16, 64, 128, 512, 1000):
                out = [C.c_int32() for _ in range(4)]
                if ((m + 15) // 16) * ((n + 15) // 16) > (1 << 31) - 1:
                    continue
                assert L.lib.sp_gemm_config(dtype, m, n, k, *[C.byref(o) for o in out]) == 0
                bm, bn, _, threads = [o.value for o in out]
                assert -(-m // bm) * -(-n // bn) * threads < 1 << 32, (m, n, k, bm, bn, threads)


def test_a_batch_adds_up_like_a_launch_per_member(L):
    """Split-K or workgroup tiles is a matter of one member's shape, for f32 always, for 16-bit inputs unless the other kind
    is estimated to be a quarter faster (large batches).  Shapes around the edges of tiles, of the K rule and of the estimate."""
    import random
    def config(dtype, m, n, k, e):
        out = [C.c_int32() for _ in range(5)]
        assert L.lib.sp_gemm_batched_config(dtype, m, n, k, e, *[C.byref(o) for o in out]) == 0
        return [o.value for o in out]
    rng = random.Random(3)
    shapes = [(0, 1536, 64, 256), (0, 64, 64, 64), (0, 128, 128, 192), (2, 1536, 128, 512), (0, 336, 304, 2256), (1, 86, 61, 56)]
    for _ in range(3000):
        dtype = rng.choice([0, 1, 2])
        m, n = (max(1, int(2 ** rng.uniform(0, 13)) // a * a) for a in (rng.choice([1, 16, 64]), rng.choice([1, 4, 64])))
        shapes.append((dtype, m, n, max(8, int(2 ** rng.uniform(3, 13)) // 8 * 8)))
    kinds, alike = {0: 0, 1: 0, 4: 0}, {e: [] for e in (2, 4, 16, 33, 64, 65, 100, 300)}
    for dtype, m, n, k in shapes:
        one = config(dtype, m, n, k, 1)
        single = [C.c_int32() for _ in range(4)]
        assert L.lib.sp_gemm_config(dtype, m, n, k, *[C.byref(o) for o in single]) == 0 and [o.value for o in single] == one[:4]
        kinds[one[4]] += 1
        for e in alike:
            many = config(dtype, m, n, k, e)
            assert dtype != 0 or many[4] == one[4], (m, n, k, e, one, many)
            alike[e].append(many[4] == one[4])
    assert kinds[1] > 300 and kinds[4] > 300
    share = lambda e: sum(alike[e]) / len(alike[e])
    assert share(2) > 0.95 and share(16) > 0.85, {e: share(e) for e in alike}
    assert L.lib.sp_gemm_batched_config(0, 64, 64, 64, 0, *[C.byref(C.c_int32()) for _ in range(5)]) == -2
    assert L.lib.sp_gemm_batched_config(0, 64, 64, 64, 2, None, *[C.byref(C.c_int32()) for _ in range(4)]) == -1


def test_batched_gemm_argument_errors(L):
    lib = L.lib
    p = C.c_void_p(0x1000)
    call = lambda **kw: lib.sp_gemm_abt_batched(0, 0, p, p, p, None, 64, 64, 64, kw.get("batch", 4), kw.get("sa", 0),
                                                kw.get("sb", 4096), kw.get("sc", 4096), 1.0, 0.0, 0, None)
    assert call(batch=0) == -2 and call(batch=70000) == -2
    assert call(sc=100) == -5 and "overlap" in _err(L)
    assert call(sb=4097) == -3
    assert call(sa=-4) == -3
    assert lib.sp_gemm_abt_batched(0, 0, None, p, p, None, 64, 64, 64, 2, 0, 4096, 4096, 1.0, 0.0, 0, None) == -1


def test_row_argument_errors(L):
    lib = L.lib
    p = C.c_void_p(0x2000)
    assert lib.sp_row_ops(None, None, None, None, None, None, None, None, 8, 8, 0, None) == -1
    assert lib.sp_row_ops(p, None, None, None, None, None, None, None, 8, 6, 0, None) == -2
    assert lib.sp_row_ops(p, None, None, None, None, None, None, None, 8, 2048, 0, None) == -2
    assert lib.sp_row_ops(p, None, None, None, None, None, None, None, 0, 8, 0, None) == -2
    assert lib.sp_row_ops(p, None, None, None, None, None, None, None, 8, 8, 1, None) == -5 and "flags" in _err(L)
    assert lib.sp_row_ops(p, None, None, None, None, None, None, p, 8, 8, 0, None) == -1  # sample without u
    assert lib.sp_row_ops(p, None, None, None, C.c_void_p(0x2008), None, None, None, 8, 8, 0, None) == -3
    assert lib.sp_row_map_f32(99, p, p, 8, 8, 0, None) == -5
    assert lib.sp_row_map_f32(L.ROW_MASKED_SOFTMAX, p, p, 8, 8, 0, None) == -5
    assert lib.sp_row_map_f32(L.ROW_MASKED_SOFTMAX, p, p, 8, 8, 9, None) == -5
    assert lib.sp_row_map_i32(L.ROW_SOFTMAX, p, p, 8, 8, None) == -5
    ph = L.PhiloxConfig(1, 0, L.PHILOX_BLOCK, 256, 24, 0, 0, 0)
    assert lib.sp_row_sample(L.ROW_SOFTMAX, p, None, None, None, None, None, p, None, 8, 8, 0, None) == -5
    assert lib.sp_row_sample(L.ROW_SOFTMAX, p, p, C.byref(ph), None, None, None, p, None, 8, 8, 0, None) == -5
    assert lib.sp_row_sample(L.ROW_LN_L2, p, p, None, None, None, None, p, None, 8, 8, 0, None) == -5
    bad = L.PhiloxConfig(1, 0, L.PHILOX_BLOCK, 100, 24, 0, 0, 0)  # 100 threads is not a multiple of cols/4 = 16
    assert lib.sp_row_sample(L.ROW_SOFTMAX, p, None, C.byref(bad), None, None, None, p, None, 8, 64, 0, None) == -5
    layer = L.PhiloxConfig(1, 0, L.PHILOX_LAYER, 256, 24, 3, 0, 0)  # 3 rows per block do not divide 8 rows
    assert lib.sp_row_sample(L.ROW_SOFTMAX, p, None, C.byref(layer), None, None, None, p, None, 8, 64, 0, None) == -5
    members = L.PhiloxConfig(1, 0, L.PHILOX_LAYER, 256, 24, 2, 3, 16)   # runs of 3 rows do not divide 8 rows
    assert lib.sp_row_sample(L.ROW_SOFTMAX, p, None, C.byref(members), None, None, None, p, None, 8, 64, 0, None) == -5
    assert lib.sp_row_get_prob(L.ROW_IDENTITY, p, None, p, 8, 8, 0, None) == -1
    assert lib.sp_row_get_prob(L.ROW_INCLUSIVE_SCAN, p, p, p, 8, 8, 0, None) == -5
    assert lib.sp_row_get_prob(L.ROW_MASKED_REGRET_MATCHING, p, p, p, 8, 8, 0, None) == -5
    assert lib.sp_row_binarize(p, p, 8, 8, 0, None) == -5 and "modulo" in _err(L)
    assert lib.sp_row_binarize(p, None, 8, 8, 7, None) == -1
    assert lib.sp_cem_resample(p, p, None, p, 8, 8, 0.1, 1.0, None) == -1
    assert lib.sp_cem_resample(p, p, p, p, 8, 6, 0.1, 1.0, None) == -2
    assert lib.sp_cem_resample_philox(p, p, 1, 0, None, 8, 8, 0.1, 1.0, None) == -1
    assert lib.sp_cem_resample_philox(p, p, 1, 6, p, 8, 8, 0.1, 1.0, None) == -5 and "multiple of 4" in _err(L)
    assert lib.sp_cem_resample_philox(p, p, 1, 0, p, 8, 6, 0.1, 1.0, None) == -2
    assert lib.sp_row_reduce_f32(0, 0, 0, p, None, 8, 8, None) == -1
    assert lib.sp_row_reduce_f32(0, 0, 0, p, p, 8, 6, None) == -2
    assert lib.sp_row_reduce_f32(9, 0, 0, p, p, 8, 8, None) == -5
    assert lib.sp_row_reduce_f32(0, 5, 0, p, p, 8, 8, None) == -5
    assert lib.sp_row_reduce_f32(0, 0, 2, p, p, 8, 8, None) == -5
    assert lib.sp_cem_update_mask(p, p, 0, None) == -2
    assert lib.sp_cem_update_mask(None, p, 4, None) == -1


def test_misc_argument_errors(L):
    lib = L.lib
    p = C.c_void_p(0x3000)
    assert lib.sp_map_f32(0, p, p, 6, None) == -2
    assert lib.sp_map_f32(0, None, p, 8, None) == -1
    assert lib.sp_reduce_sum(0, p, p, 8, p, 16, None) == -5
    big = lib.sp_reduce_workspace_bytes()
    assert lib.sp_reduce(4, 0, p, p, 8, p, big, None) == -5 and "op must be" in _err(L)     # no whole-tensor average
    assert lib.sp_reduce(2, 3, p, p, 8, p, big, None) == -4
    assert lib.sp_reduce(2, 0, p, p, 0, p, big, None) == -2
    assert lib.sp_reduce(2, 0, p, p, 8, None, big, None) == -1
    assert lib.sp_reduce_status(p, 16, C.byref(C.c_int64()), None) == -5
    assert lib.sp_reduce_status(p, big, None, None) == -1
    assert lib.sp_reduce_set_poll_limit(20000000) == -5 and lib.sp_reduce_set_poll_limit(0) == 0
    assert lib.sp_row_l1_normalize(p, p, 4, 8, 0.0, None) == -5 and "threshold" in _err(L)
    assert lib.sp_row_l1_normalize(p, None, 4, 8, 1.0, None) == -1
    assert lib.sp_reduce_workspace_bytes() >= 1024
    assert lib.sp_transpose_inner_b32(p, p, 1, 8, 8, None) == -5
    assert lib.sp_transpose_inner_b32(p, C.c_void_p(0x4000), 0, 8, 8, None) == -2
    assert lib.sp_device_info(None) == -1


def test_mlp_argument_errors(L):
    lib = L.lib
    p = C.c_void_p(0x5000)
    w = (C.c_void_p * 2)(p, p)
    dims = lambda *d: (C.c_int32 * len(d))(*d)
    call = lambda dtype=1, x=p, n=2, ws=w, d=dims(32, 64, 3), u=None, ph=None, pol=p, act=None, batch=8, head=3, mask=0: \
        lib.sp_mlp_forward(dtype, x, n, ws, None, d, u, ph, pol, act, None, batch, head, mask, None)
    assert call(dtype=0) == -4
    assert call(x=None) == -1
    assert call(n=0) == -5 and call(n=9) == -5
    assert call(d=dims(30, 64, 3)) == -2
    assert call(d=dims(32, 48, 3)) == -2
    assert call(d=dims(32, 512, 3)) == -2
    assert call(d=dims(32, 64, 128)) == -2
    assert call(batch=0) == -2
    assert call(head=7) == -5
    assert call(mask=4) == -5
    assert call(act=p) == -1  # action without u
    assert call(ws=(C.c_void_p * 2)(p, None)) == -1
    # a head that draws its own uniforms: one of u / philox, and the output width must be a row width of the
    # reference's sampling op (a multiple of 4) whose 4-column thread groups divide the block
    ph = L.PhiloxConfig(12344321, 0, L.PHILOX_LAYER, 256, 24, 8, 0, 0)
    assert call(act=p, u=p, ph=C.byref(ph)) == -5 and "at most one" in _err(L)
    assert call(act=p, ph=C.byref(ph)) == -5 and "multiple of 4" in _err(L)
    assert call(act=p, ph=C.byref(ph), d=dims(32, 64, 64), batch=24 * 8 + 1) == -5 and "rows_per_block" in _err(L)
    bad = L.PhiloxConfig(12344321, 0, 9, 256, 24, 8, 0, 0)
    assert call(act=p, ph=C.byref(bad), d=dims(32, 64, 64)) == -5 and "philox mode" in _err(L)


def test_packed_mlp_argument_errors(L):
    lib = L.lib
    p = C.c_void_p(0x6000)
    dims = lambda *d: (C.c_int32 * len(d))(*d)
    assert lib.sp_mlp_packed_bytes(4, dims(32, 256, 256, 256, 3)) == 4 * 4096 + 2 * 131072 + 8192
    assert lib.sp_mlp_packed_bytes(3, dims(128, 256, 256, 64)) == 4 * 8 * 4096 + 131072 + 8192
    assert lib.sp_mlp_packed_bytes(3, dims(32, 128, 256, 3)) == 0
    assert lib.sp_mlp_packed_bytes(2, dims(32, 256, 3)) == 0
    assert lib.sp_mlp_packed_bytes(6, dims(32, 256, 256, 256, 256, 256, 3)) == 0
    assert lib.sp_mlp_packed_bytes(4, None) == 0
    w = (C.c_void_p * 4)(p, p, p, p)
    d = dims(32, 256, 256, 256, 3)
    assert lib.sp_mlp_pack_weights(1, 4, w, d, None, 1 << 20, None) == -1
    assert lib.sp_mlp_pack_weights(0, 4, w, d, p, 1 << 20, None) == -4
    assert lib.sp_mlp_pack_weights(1, 4, w, d, p, 1000, None) == -5 and "must hold" in _err(L)
    assert lib.sp_mlp_pack_weights(1, 4, w, dims(32, 256, 128, 256, 3), p, 1 << 20, None) == -6
    assert lib.sp_mlp_pack_weights(1, 4, (C.c_void_p * 4)(p, None, p, p), d, p, 1 << 20, None) == -1
    size = lib.sp_mlp_packed_bytes(4, d)
    call = lambda dtype=1, x=p, n=4, pk=p, nbytes=size, dd=d, u=None, pol=p, act=None, logits=None, batch=8, head=1, mask=0: \
        lib.sp_mlp_forward_packed(dtype, x, n, pk, nbytes, None, dd, u, None, pol, act, logits, batch, head, mask, None)
    # a buffer packed for another stack (another layer count, another class of first width) has another size
    assert call(nbytes=lib.sp_mlp_packed_bytes(3, dims(32, 256, 256, 3))) == -5 and "another stack" in _err(L)
    assert call(nbytes=lib.sp_mlp_packed_bytes(4, dims(64, 256, 256, 256, 3))) == -5
    assert call(nbytes=size + 16) == -5
    assert call(dtype=0) == -4
    assert call(pk=None) == -1
    assert call(batch=0) == -2
    assert call(act=p) == -1                                        # action without u
    assert call(dd=dims(32, 256, 64, 256, 3)) == -6                 # a hidden width other than 256
    assert call(dd=dims(32, 256, 256, 256, 64)) == -6 and "16 outputs" in _err(L)     # wide head, no mask
    assert call(dd=dims(32, 256, 256, 256, 64), mask=3, logits=p) == -6               # wide masked head with logits
    assert call(mask=4) == -5


def test_ensemble_argument_errors(L):
    lib = L.lib
    p = C.c_void_p(0x6000)
    dims = lambda *d: (C.c_int32 * len(d))(*d)
    w2 = (C.c_void_p * 2)(p, p)
    call = lambda dtype=0, x=p, n=2, w=w2, dd=dims(128, 64, 64), members=4, u=None, pol=p, act=None, batch=64, head=2, mask=3: \
        lib.sp_mlp_forward_ensemble(dtype, x, n, w, dd, members, u, None, pol, act, batch, head, mask, None)
    assert call(dtype=1) == -4                                       # f32 only
    assert call(x=None) == -1 and call(pol=None) == -1 and call(w=None) == -1
    assert call(n=3) == -2 and "one or two layers" in _err(L)
    assert call(dd=dims(128, 32, 64)) == -2 and "hidden width" in _err(L)
    assert call(dd=dims(136, 64, 64)) == -2                         # two layers: inputs up to 128 wide
    assert call(dd=dims(20, 64, 64)) == -2                          # a multiple of 8
    assert call(mask=0) == -2 and "at most 4 computed outputs" in _err(L)
    assert call(mask=65) == -5
    assert call(members=0) == -2 and call(batch=0) == -2
    assert call(act=p) == -1                                        # an action without uniforms
    assert call(w=(C.c_void_p * 2)(p, None)) == -1
    assert call(x=C.c_void_p(0x6004)) == -3
    # one layer: inputs up to 256 wide, the same head limits
    one = (C.c_void_p * 1)(p)
    assert call(n=1, w=one, dd=dims(264, 64)) == -2
    assert call(n=1, w=one, dd=dims(256, 64), mask=5) == -2
    hash_call = lambda dtype=0, x=p, w=p, out=p, members=4, batch=64, k0=128, n=128, modulo=4096: \
        lib.sp_ensemble_binarize(dtype, x, w, out, members, batch, k0, n, modulo, None)
    assert hash_call(dtype=2) == -4
    assert hash_call(x=None) == -1 and hash_call(w=None) == -1 and hash_call(out=None) == -1
    assert hash_call(k0=260) == -2 and hash_call(k0=12) == -2 and hash_call(n=0) == -2
    assert hash_call(modulo=0) == -5 and "modulo" in _err(L)
    assert hash_call(members=70000) == -2
    assert hash_call(w=C.c_void_p(0x6008)) == -3


def test_stack_argument_errors(L):
    p = C.c_void_p(0x6000)
    ints = lambda *d: (C.c_int32 * len(d))(*d)
    call = lambda x=p, n=2, w=(C.c_void_p * 2)(p, p), d=ints(64, 64, 16), acts=ints(1, 0), members=1, pol=p, act=None, batch=64, head=1, mask=0, ph=None: \
        L.lib.sp_stack_forward_f32(x, n, w, d, acts, members, None, ph, pol, act, batch, head, mask, None)
    assert call(x=None) == -1 and call(pol=None) == -1 and call(w=None) == -1 and call(w=(C.c_void_p * 2)(p, None)) == -1
    assert call(act=p) == -1                                          # an action without uniforms
    assert call(x=C.c_void_p(0x6004)) == -3
    assert call(n=9) == -2 and call(members=0) == -2 and call(batch=0) == -2 and call(batch=1 << 31) == -2
    assert call(d=ints(66, 64, 16)) == -2 and call(d=ints(64, 72, 16)) == -2 and call(d=ints(64, 64, 68)) == -2 and call(d=ints(64, 144, 16)) == -2
    assert call(head=3) == -5 and call(acts=ints(9, 0)) == -5 and call(head=2, mask=0) == -5 and call(head=2, mask=17) == -5
    ph = L.PhiloxConfig(1, 0, L.PHILOX_LAYER, 256, 8, 8, 32, 0)
    assert call(act=p, ph=C.byref(ph)) == -5 and "member_rows" in _err(L)
    assert call(n=4, w=(C.c_void_p * 4)(p, p, p, p), d=ints(128, 128, 128, 128, 64), acts=ints(1, 1, 1, 0)) == -6 and "LDS" in _err(L)


def test_a_stack_reads_no_activation_behind_its_last_layer(L):
    """acts holds n_layers - 1 codes: what lies behind them is not looked at (here a code that is refused anywhere else, in a call
    that is refused for its random stream, so nothing is launched)."""
    p = C.c_void_p(0x6000)
    ints = lambda *d: (C.c_int32 * len(d))(*d)
    stream = L.PhiloxConfig(1, 0, L.PHILOX_LAYER, 256, 8, 8, 32, 0)      # member_rows is not the batch
    call = lambda *acts: L.lib.sp_stack_forward_f32(p, 2, (C.c_void_p * 2)(p, p), ints(64, 64, 16), ints(*acts), 1, None,
                                                    C.byref(stream), p, p, 64, 1, 0, None)
    assert call(1, 9) == -5 and "member_rows" in _err(L)
    assert call(9, 0) == -5 and "activation" in _err(L)


def test_stack_sizes_are_asked_without_a_call(L):
    ints = lambda *d: (C.c_int32 * len(d))(*d)
    takes = lambda *d, members=1, batch=64, head=1, mask=0: L.lib.sp_stack_forward_takes(len(d) - 1, ints(*d), members, batch, head, mask)
    assert takes(64, 64, 64, 64) == 0 and takes(4, 16, 4) == 0 and takes(128, 128, 128, 64) == -6 and takes(128, 128, 128, 64, head=2, mask=16) == 0
    assert takes(66, 64, 16) == -2 and takes(64, 72, 16) == -2 and takes(64, 144, 16) == -2 and takes(64, 64, 68) == -2
    assert takes(64, 16, members=70000) == -2 and takes(64, 16, batch=0) == -2 and takes(64, 16, members=2, batch=1 << 30) == -2
    assert takes(64, 16, head=3) == -5 and takes(64, 16, head=2, mask=17) == -5 and takes(*([64] * 10)) == -2
    assert L.lib.sp_stack_forward_takes(1, None, 1, 64, 1, 0) == -1


@pytest.mark.parametrize("m,n,k", [(13040, 96, 5112), (5168, 224, 5048), (1732, 943, 5784), (24937, 56, 8088), (3584, 592, 2296), (16512, 96, 1000)])
def test_long_k_of_one_round_is_not_left_to_lone_workgroups(L, m, n, k):
    """16-bit shapes of at most one 128 x 96 tile per compute unit of 256, where nothing covers such a workgroup's loads."""
    for dtype in (1, 2):
        out = [C.c_int32() for _ in range(4)]
        assert L.lib.sp_gemm_config(dtype, m, n, k, *[C.byref(o) for o in out]) == 0
        assert (out[0].value, out[1].value) != (128, 96)


@pytest.mark.parametrize("m,n,k", [(53584, 16, 272), (51392, 16, 120), (60000, 32, 200)])
def test_tiles_that_are_half_padding_are_not_taken_for_whole_pieces(L, m, n, k):
    out = [C.c_int32() for _ in range(4)]
    assert L.lib.sp_gemm_config(1, m, n, k, *[C.byref(o) for o in out]) == 0
    assert out[1].value <= 64 and (out[0].value, out[1].value) != (128, 64)
