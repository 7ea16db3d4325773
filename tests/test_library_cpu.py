"""CPU-side checks of the product: the C-ABI libraries load and export every declared symbol,
the host workload generator matches published SplitMix64/FNV values and the oracle's encoders,
and the byte accounting matches the benchmark definition.  No GPU calls."""

import ctypes
import os
import re

import numpy as np
import pytest

from urbilateria_amd import configs as C
from urbilateria_amd import native as N
from urbilateria_amd import synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared(header):
    text = open(os.path.join(ROOT, "include", header)).read()
    return sorted(set(re.findall(r"\b(urb_[a-z0-9_]+)\s*\(", text)))


def test_moe_library_exports_every_declared_symbol():
    lib = ctypes.CDLL(N.MOE_LIB)
    declared = _declared("urb_moe.h")
    assert declared, "no declarations found"
    for name in declared:
        assert hasattr(lib, name), name
    assert set(N.EXPORTS) == set(declared)


def _prototypes(header):
    text = re.sub(r"/\*.*?\*/", "", open(os.path.join(ROOT, "include", header)).read(),
                  flags=re.S)
    out = {}
    for name, params in re.findall(r"\b(urb_\w+)\s*\(([^;{]*?)\)\s*;", text, flags=re.S):
        ps = [p.strip() for p in params.replace("\n", " ").split(",")]
        out[name] = [p for p in ps if p and p != "void"]
    return out


_SCALARS = {"uint32_t": ctypes.c_uint32, "int": ctypes.c_int, "float": ctypes.c_float,
            "urb_format": ctypes.c_int, "urb_weight_source": ctypes.c_int,
            "urb_status": ctypes.c_int}


def test_moe_bindings_match_the_header_prototypes():
    # Every ctypes binding passes each parameter as the header declares it: pointers as
    # pointer-sized values, scalars as their C type (a pointer bound as an int would be cut to
    # 32 bits).
    lib = N.moe_lib()
    protos = _prototypes("urb_moe.h")
    assert set(protos) == set(N.EXPORTS)
    for name, params in protos.items():
        at = getattr(lib, name).argtypes
        assert at is not None and len(at) == len(params), name
        for p, t in zip(params, at):
            if "*" in p:
                assert t is ctypes.c_void_p or issubclass(t, ctypes._Pointer), (name, p, t)
            else:
                ctype = p.replace("const ", "").rsplit(" ", 1)[0].strip()
                assert t is _SCALARS[ctype], (name, p, t)


def test_synth_library_exports():
    lib = ctypes.CDLL(N.SYNTH_LIB)
    for name in N.SYNTH_EXPORTS:
        assert hasattr(lib, name), name


def test_status_strings():
    lib = N.moe_lib()
    for s in range(8):
        assert lib.urb_status_string(s)


def test_splitmix64_published_vectors():
    # SplitMix64 (Steele, Lea, Flood 2014) seeded with 0; the reference's generator
    # (src/generation.rs:419-440) uses the same constants.
    got = [int(v) for v in synth.splitmix64(0, 0, 3)]
    assert got == [0xE220A8397B1DCDAF, 0x6E789E6AA1B965F4, 0x06C45D188009454F]
    # counter form: draw n of seed s equals draw 0 of seed s + n * gamma
    a = synth.splitmix64(12345, 7, 1)[0]
    b = synth.splitmix64((12345 + 7 * 0x9E3779B97F4A7C15) & (2**64 - 1), 0, 1)[0]
    assert a == b


def test_fnv1a64_published_vectors():
    assert synth.fnv1a64("") == 0xCBF29CE484222325
    assert synth.fnv1a64("a") == 0xAF63DC4C8601EC8C
    assert synth.fnv1a64("foobar") == 0x85944171F73967E8


def test_host_encoders_agree_with_oracle():
    from oracle import oracle as O
    rng = np.random.default_rng(11)
    vals = np.concatenate([rng.standard_normal(3000).astype(np.float32) * 60,
                           rng.standard_normal(500).astype(np.float32) * 1e-3,
                           np.array([0.0, -0.0, 448.0, -448.0, 1000.0, -1e9], np.float32)])
    codes = synth.encode_e4m3fn(vals)
    for v, c in zip(vals, codes):
        assert int(c) == O.encode_e4m3fn_finite(float(v)), v
    bits = synth.bf16_rne_bits(vals[:3000])
    for v, b in zip(vals[:3000], bits):
        assert (np.uint32(b) << np.uint32(16)).view(np.float32) == O.round_to_bf16(float(v))


def test_generator_distributions():
    z = synth.normals(synth.stream_seed("x"), 200000)
    assert abs(float(z.mean())) < 0.01 and abs(float(z.std()) - 1.0) < 0.01
    p, s = synth.mxfp4_matrix("m", 64, 256)
    nib = np.concatenate([p & 15, p >> 4]).ravel()
    assert set(np.unique(nib)) == set(range(16))
    assert s.min() >= 119 and s.max() <= 125 and s.shape == (64, 8)
    c, s8 = synth.mxfp8_matrix("m8", 16, 64)
    assert not np.any((c & 0x7F) == 0x7F)


def test_benchmark_byte_accounting():
    W = C.WORKLOADS
    assert C.expert_bytes(W["c1_bf16_decode"].spec) == 9_437_184
    assert C.expert_bytes(W["c3_mxfp4_decode"].spec) == 23_396_352
    assert C.expert_bytes(W["c4_mxfp8"].spec) == 38_928_384
    assert C.shared_bytes(W["c3_mxfp4_decode"].spec) == 88_080_384


def test_synthetic_hash_table_rows_are_distinct_in_range_and_seeded():
    for vocab, E, k in ((129280, 256, 6), (50, 32, 6), (40, 24, 8), (7, 6, 6), (3, 1, 1)):
        t = C.hash_table(vocab, E, k)
        assert t.shape == (vocab, k) and t.dtype == np.int64
        assert t.min() >= 0 and t.max() < E
        srt = np.sort(t, axis=1)
        assert not np.any(srt[:, 1:] == srt[:, :-1])  # distinct within each row
        assert np.array_equal(t, C.hash_table(vocab, E, k))
    assert not np.array_equal(C.hash_table(50, 32, 6), C.hash_table(50, 32, 6, base_seed=7))
    w = C.workload("dsv4_flash_hash")
    assert w.hash_vocab == 129280 and w.spec.composition == C.COMPOSE_DSV4
    assert C.workload("dsv4_flash").spec.top_k == 6


def test_zipf_bias_is_monotone_in_rank():
    b = C.zipf_bias(384, 1.1, 0.1)
    assert b.shape == (384,) and np.all(np.isfinite(b))
    assert len(np.unique(b)) == 384


def _inclusion_by_enumeration(p, k):
    """Inclusion probabilities of successive sampling by summing every ordered k-draw."""
    import itertools
    p = np.asarray(p, np.float64) / np.sum(p)
    pi = np.zeros(len(p))
    for seq in itertools.permutations(range(len(p)), k):
        pr, rest = 1.0, 1.0
        for e in seq:
            pr *= p[e] / rest
            rest -= p[e]
        pi[list(seq)] += pr
    return pi


@pytest.mark.parametrize("E,k", [(5, 1), (5, 2), (6, 3), (7, 4), (4, 4)])
def test_zipf_inclusion_equals_enumeration(E, k):
    # brute force over all ordered draws; k = 1 is p itself, k = E is all ones
    p = np.linspace(1.0, 0.05, E) ** 3
    got = C.zipf_inclusion(p, k)
    ref = _inclusion_by_enumeration(p, k)
    assert np.allclose(got, ref, atol=1e-6), (got, ref)
    assert abs(got.sum() - k) < 1e-5
    if k == 1:
        assert np.allclose(got, p / p.sum(), atol=1e-6)


def test_selection_bias_fit_meets_its_targets():
    # i.i.d. U(0, 1) scores over 12 experts, top-3: the fitted bias must reproduce any
    # feasible marginals, here a geometric popularity profile
    u = synth.unit_f64(synth.splitmix64(synth.stream_seed("test.fit"), 0, 4000 * 12))
    scores = u.reshape(4000, 12)
    pi = C.zipf_inclusion(0.7 ** np.arange(12), 3)
    bias, counts = C.fit_selection_bias(scores, 3, 4000 * pi)
    assert counts.sum() == 4000 * 3
    assert np.abs(counts - 4000 * pi).max() <= 3, (counts, 4000 * pi)
    # the counts are the top-3 of the biased scores
    top = np.argsort(-(scores + bias[None, :]), axis=1, kind="stable")[:, :3]
    assert np.array_equal(np.bincount(top.ravel(), minlength=12), counts)
    assert np.all(np.diff(bias[np.argsort(-pi)]) <= 1e-9)  # more popular, larger bias


def test_c5_bias_gives_zipf_top8_marginals():
    # the headline's per-expert bias: the hottest expert at its inclusion probability under
    # Zipf(1.1) top-8 without replacement (0.854), on the calibration draw and on the
    # benchmark's own 1024 tokens through the seeded router
    w = C.workload("c5_mxfp4_zipf_prefill")
    info, bias = C.workload_bias(w)
    assert info["fit"] == "marginals" and abs(info["target_top_share"] - 0.8544) < 1e-3
    assert info["max_abs_count_error"] <= 8
    spec = w.spec
    router = synth.bf16_to_f32(synth.bf16_matrix("router", spec.n_experts, spec.hidden, 0.02))
    x = synth.activations("x", 1024, spec.hidden)
    g = C.router_scores(spec.router, (x.astype(np.float64) @ router.T.astype(np.float64)))
    top = np.argpartition(-(g + bias[None, :]), spec.top_k - 1, axis=1)[:, :spec.top_k]
    counts = np.bincount(top.ravel(), minlength=spec.n_experts)
    assert 800 <= counts.max() <= 900 and (counts > 0).sum() >= 360, (counts.max(),
                                                                      (counts > 0).sum())


@pytest.mark.parametrize("fmt", [C.FMT_BF16, C.FMT_MXFP4, C.FMT_MXFP8])
def test_expert_views_slice_consolidated_tensors(fmt):
    # urb_expert_views only computes addresses, so host tensors stand in for device ones.  The
    # views must be the per-expert slices the reference takes: gate = rows 0..I-1 and up = rows
    # I..2I-1 of each expert's [2I, H] block, down = the expert's [H, I] block, with the scale
    # sidecars sliced the same way (qwen3_6/expert_store.rs:146-158, hy4/expert.rs:664-680).
    torch = pytest.importorskip("torch")
    from urbilateria_amd import moe
    E, H, I = 3, 256, 128
    spec = C.LayerSpec(hidden=H, n_experts=E, top_k=2, intermediate=I, expert_format=fmt)
    width = {C.FMT_BF16: 2 * H, C.FMT_MXFP4: H // 2, C.FMT_MXFP8: H}[fmt]
    dwidth = {C.FMT_BF16: 2 * I, C.FMT_MXFP4: I // 2, C.FMT_MXFP8: I}[fmt]
    gu = torch.zeros((E, 2 * I, width), dtype=torch.uint8)
    dn = torch.zeros((E, H, dwidth), dtype=torch.uint8)
    mx = fmt != C.FMT_BF16
    gus = torch.zeros((E, 2 * I, H // 32), dtype=torch.uint8) if mx else None
    dns = torch.zeros((E, H, I // 32), dtype=torch.uint8) if mx else None
    layer = moe.DeviceLayer.from_consolidated(spec, None, gu, gus, dn, dns)
    views = moe.expert_views(fmt, E, H, I, gu, gus, dn, dns)
    for e in range(E):
        for m in range(3):
            d, s = layer.experts[e][m]
            assert d.is_contiguous() and (s is None or s.is_contiguous())
            assert views[3 * e + m] == (d.data_ptr(), None if s is None else s.data_ptr())
    # the up view starts one [I, H] matrix after the gate view
    row = C.matrix_bytes(fmt, I, H)[0]
    assert views[1][0] - views[0][0] == row
    assert views[3][0] - views[0][0] == 2 * row


def test_expert_views_rejects_bad_arguments():
    lib = N.moe_lib()
    out = (N.Matrix * 3)()
    a = ctypes.addressof(out)
    # BF16 takes no scales; MX formats need both scale tensors
    assert lib.urb_expert_views(C.FMT_BF16, 1, 256, 128, 16, 16, 16, None, a) == N.ERR_ARGUMENT
    assert lib.urb_expert_views(C.FMT_MXFP4, 1, 256, 128, 16, 16, 16, None, a) == N.ERR_ARGUMENT
    assert lib.urb_expert_views(C.FMT_MXFP8, 1, 250, 128, 16, 16, 16, 16, a) == N.ERR_SHAPE
    assert lib.urb_expert_views(C.FMT_BF16, 0, 256, 128, 16, None, 16, None, a) == N.ERR_ARGUMENT
    assert lib.urb_expert_views(C.FMT_BF16, 1, 256, 128, 16, None, 16, None, a) == N.OK


def _placement(fmt, pair, dense, tiles, rows, cols):
    lib = N.moe_lib()
    n = lib.urb_gemm_placement(fmt, pair, dense, tiles, rows, cols, None, None, 0)
    assert n > 0
    t = np.empty(n, np.int32)
    g = np.empty(n, np.int32)
    assert lib.urb_gemm_placement(fmt, pair, dense, tiles, rows, cols, t.ctypes.data,
                                  g.ctypes.data, n) == n
    return t, g


def _groups(fmt, rows, pair, dense):
    if fmt == C.FMT_BF16:
        np_ = 1 if dense <= 64 else (4 if not pair and rows % 256 == 0 else 2)
    elif fmt == C.FMT_MXFP8:
        np_ = 4 if not pair and rows % 256 == 0 else 2
    else:
        np_ = 2 if pair else 4 if rows % 256 == 0 else 2
    return rows // (64 * np_)


@pytest.mark.parametrize("fmt,rows,cols", [(C.FMT_BF16, 2048, 7168), (C.FMT_BF16, 7168, 2048),
                                           (C.FMT_MXFP4, 2048, 7168), (C.FMT_MXFP4, 7168, 2048),
                                           (C.FMT_MXFP4, 4224, 2048), (C.FMT_MXFP8, 6144, 2048),
                                           (C.FMT_BF16, 768, 2048), (C.FMT_MXFP8, 768, 2048),
                                           (C.FMT_MXFP8, 2048, 768)])
def test_grouped_gemm_placement_covers_every_pair_once_and_every_xcd(fmt, rows, cols):
    # The grouped GEMM's workgroup -> (row tile, panel group) mapping, replayed on the host from
    # the same placement function the kernel runs: every (tile, group) pair is computed by
    # exactly one workgroup, and (workgroups go to the XCDs round robin, block % 8) every XCD
    # has work -- for a dense batch (the shared expert) of any size, where one or two tiles
    # used to land on one XCD, and for routed tile lists of any length >= 8.  (Tall-tile launches of
    # every format, BF16 too, are placed as MXFP8's of the same rows.)
    cases = [(T, (T + 31) // 32) for T in list(range(1, 65)) + [96, 128, 200, 256, 1024]]
    cases += [(0, n) for n in (8, 9, 13, 40, 163, 550)]
    for dense, tiles in cases:
        for pair in (0, 1):
            groups = _groups(fmt, rows, pair, dense)
            t, g = _placement(fmt, pair, dense, tiles, rows, cols)
            work = t >= 0
            pairs = list(zip(t[work].tolist(), g[work].tolist()))
            assert len(pairs) == len(set(pairs)) == tiles * groups, (dense, tiles)
            assert set(pairs) == {(a, b) for a in range(tiles) for b in range(groups)}
            if groups >= 8 or tiles >= 8:
                xcds = set((np.nonzero(work)[0] % 8).tolist())
                assert xcds == set(range(8)), (dense, tiles, pair, sorted(xcds))


def _meta(dtype, shape, elem=1):
    n = int(np.prod(shape)) * elem
    return {"dtype": dtype, "shape": list(shape), "data_len": n}


def test_inspect_matrix_selects_formats_from_metadata_like_the_reference():
    # inspect_weight_matrix (src/storage/weight.rs:118-330): the reference's own fixtures --
    # Kimi native MXFP4 `expert.w1.weight_packed` U8 [2, 1] + U8 scale [2, 1] -> 4 resident
    # bytes (weight.rs:1035-1053); ModelOpt MXFP8 E4M3 [2, 33] + U8 [2, 2] -> 70 bytes
    # (weight.rs:1056-1077) -- then DeepSeek-style I8 + F8_E8M0 MXFP4 and plain BF16
    F = N.inspect_matrix
    assert F(_meta("U8", (2, 1)), _meta("U8", (2, 1)), 2, 2, packed_name=True) == (C.FMT_MXFP4, 4)
    assert F(_meta("F8_E4M3", (2, 33)), _meta("U8", (2, 2)), 2, 33) == (C.FMT_MXFP8, 70)
    assert F(_meta("I8", (2048, 3584)), _meta("F8_E8M0", (2048, 224)), 2048, 7168) == \
        (C.FMT_MXFP4, 2048 * 3584 + 2048 * 224)
    # plain BF16 [2, 2]: compact BF16, 8 resident bytes -- inspect_compact_bf16_matrix's answer
    # for the reference's fixture (weight.rs:1237-1243); inspect_weight_matrix would widen the
    # same tensor to F32, 16 bytes (weight.rs:1267-1273), which this layer never does
    assert F(_meta("BF16", (2, 2), 2), None, 2, 2) == (C.FMT_BF16, 8)


@pytest.mark.parametrize("weight,scale,rows,cols,packed,status", [
    # E4M3 with DeepSeek-V4.1 32x32 or DeepSeek-V4 128x128 E8M0 block scales: a format the
    # reference reads (MxFp8E4M3 32x32 / 128x128) that this layer does not take
    (("F8_E4M3", (64, 64)), ("F8_E8M0", (2, 2)), 64, 64, False, N.ERR_ARGUMENT),
    (("F8_E4M3", (129, 129)), ("F8_E8M0", (2, 2)), 129, 129, False, N.ERR_ARGUMENT),
    # E4M3 without a sidecar: require_mx_scale's Unsupported
    (("F8_E4M3", (2, 32)), None, 2, 32, False, N.ERR_ARGUMENT),
    # a sidecar of no known geometry, a weight of the wrong shape: InvalidShape
    (("F8_E4M3", (2, 33)), ("U8", (2, 1)), 2, 33, False, N.ERR_SHAPE),
    (("F8_E4M3", (1, 129)), ("U8", (2, 5)), 2, 129, False, N.ERR_SHAPE),
    # MXFP4: I8 payload wants an F8_E8M0 sidecar, U8 `.weight_packed` a U8 one
    (("I8", (2, 16)), ("U8", (2, 1)), 2, 32, False, N.ERR_SHAPE),
    (("U8", (2, 16)), ("F8_E8M0", (2, 1)), 2, 32, True, N.ERR_SHAPE),
    (("I8", (2, 15)), ("F8_E8M0", (2, 1)), 2, 32, False, N.ERR_SHAPE),
    # U8 not named `.weight_packed`: Colibri INT4/INT8 with an F32 sidecar, not taken here
    (("U8", (2, 16)), ("U8", (2, 1)), 2, 32, False, N.ERR_ARGUMENT),
    # plain F32 / F16 matrices, plain matrices of the wrong shape, empty matrices
    (("F32", (2, 2)), None, 2, 2, False, N.ERR_ARGUMENT),
    (("F16", (2, 2)), None, 2, 2, False, N.ERR_ARGUMENT),
    (("BF16", (2, 3)), None, 2, 2, False, N.ERR_SHAPE),
    (("BF16", (0, 2)), None, 0, 2, False, N.ERR_SHAPE),
])
def test_inspect_matrix_errors(weight, scale, rows, cols, packed, status):
    esize = {"BF16": 2, "F16": 2, "F32": 4}.get(weight[0], 1)
    w = _meta(weight[0], weight[1], esize)
    s = None if scale is None else _meta(scale[0], scale[1])
    with pytest.raises(N.UrbError) as e:
        N.inspect_matrix(w, s, rows, cols, packed_name=packed)
    assert e.value.status == status


def test_tall_down_kernels_share_row_scales_behind_a_barrier(tmp_path):
    # The f16 down projection over tall tiles leaves each row's power of two in LDS for the seven
    # other threads that stage the row: in every such kernel a workgroup barrier stands between the
    # last of those stores and the first load (LDS order within a wave is the compiler's to change).
    from urbilateria_amd import build as B
    out = tmp_path / "tall.s"
    flags = [f for f in B.HIPCC_FLAGS if f not in ("-O3", "-fPIC", "-shared")]
    B._run([B._hipcc(), *flags, "-O1", "--cuda-device-only", "-S", "-o", str(out),
            os.path.join(B.CSRC, "urb_tall.hip")])
    kernels = 0
    for body in re.split(r"\n(?=_Z\w*tall_kernel\w*:)", out.read_text())[1:]:
        if not re.match(r"_Z\w*tall_kernelILi[12]ELb0ELi1E", body):   # MXFP4, MXFP8; down; f16 rows
            continue
        kernels += 1
        ops = re.findall(r"\n\s+(ds_write2?(?:st64)?_b32|ds_read2?(?:st64)?_b32|s_barrier)\b",
                         body.split("s_endpgm")[0])
        first_read = next(i for i, op in enumerate(ops) if op.startswith("ds_read"))
        stores = [i for i, op in enumerate(ops[:first_read]) if op.startswith("ds_write")]
        assert stores and "s_barrier" in ops[stores[-1]:first_read], body.split(":")[0]
    assert kernels == 2


def _tiles(workload, tokens, **dims):
    from dataclasses import replace

    from .gpu_helpers import tile_rows
    return tile_rows(replace(C.workload(workload).spec, **dims), tokens)


@pytest.mark.parametrize("workload,per,dims,rows", [
    # tokens per expert, layer -> tokens per row tile.  Tall tiles (128) need a round of workgroups
    # (two on each of 256 CUs) in the gate/up launch: experts x tiles x intermediate / 128 >= 512 ...
    ("c2_bf16_prefill", 40, dict(n_experts=64, intermediate=1024), 128),
    ("c2_bf16_prefill", 40, dict(n_experts=64, intermediate=896), 32),
    ("c2_bf16_prefill", 39, dict(n_experts=64, intermediate=1024), 32),
    ("c2_bf16_prefill", 128, dict(n_experts=64, intermediate=512), 32),
    ("c2_bf16_prefill", 63, dict(n_experts=64, intermediate=768), 32),     # three quarters
    ("c2_bf16_prefill", 64, dict(n_experts=64, intermediate=768), 128),
    ("c2_bf16_prefill", 129, dict(n_experts=64, intermediate=512), 128),   # two tiles each
    ("qwen36_release", 60, {}, 128),                                       # 256 x 512
    ("c4_mxfp8", 36, dict(n_experts=32), 128), ("c4_mxfp8", 35, dict(n_experts=32), 32),
    # ... MXFP8 from 64 tokens per expert on half a round, MXFP4 two to four rounds by hidden size
    ("c4_mxfp8", 63, dict(n_experts=16), 32), ("c4_mxfp8", 64, dict(n_experts=16), 128),
    ("c4_mxfp8", 96, dict(n_experts=8), 32),
    ("c3_mxfp4_decode", 64, {}, 128), ("c3_mxfp4_decode", 63, {}, 32),     # 256 x 2048 of 7168
    ("c3_mxfp4_decode", 64, dict(n_experts=128), 128),
    ("c3_mxfp4_decode", 64, dict(n_experts=128, intermediate=1408), 32),
    ("c3_mxfp4_decode", 64, dict(n_experts=128, intermediate=1536), 128),
    ("c3_mxfp4_decode", 83, dict(n_experts=128, intermediate=1024), 32),
    ("c3_mxfp4_decode", 84, dict(n_experts=128, intermediate=1024), 128),
    ("c3_mxfp4_decode", 100, dict(n_experts=128, intermediate=896), 32),
    ("c3_mxfp4_decode", 64, dict(hidden=5120, n_experts=128), 128),
    ("c3_mxfp4_decode", 83, dict(hidden=5120, n_experts=128, intermediate=1920), 32),
    ("c3_mxfp4_decode", 84, dict(hidden=5120, n_experts=128, intermediate=1536), 128),
    ("c3_mxfp4_decode", 83, dict(hidden=4096), 32),
    ("c3_mxfp4_decode", 84, dict(hidden=4096), 128),
    ("c3_mxfp4_decode", 100, dict(hidden=4096, n_experts=128, intermediate=1920), 32),
    ("c3_mxfp4_decode", 100, dict(n_experts=32, intermediate=1024), 32),
    # MX activations: MXFP8 on 64-token tiles in between, MXFP4 only over four rounds
    ("c4_mxfp8_mx_activation", 31, {}, 32), ("c4_mxfp8_mx_activation", 32, {}, 64),
    ("c4_mxfp8_mx_activation", 63, {}, 64), ("c4_mxfp8_mx_activation", 64, {}, 128),
    ("c4_mxfp8_mx_activation", 40, dict(n_experts=16, intermediate=1024), 32),
    ("c4_mxfp8_mx_activation", 100, dict(n_experts=16, intermediate=1024), 32),
    ("dsv4_flash", 95, {}, 32),                                            # 256 x 2048
    ("dsv4_flash", 127, dict(n_experts=128), 32), ("dsv4_flash", 128, dict(n_experts=128), 128),
    ("dsv4_flash", 128, dict(n_experts=96, intermediate=1024), 32),
    # tall down projections take 256 rows at a time
    ("c4_mxfp8", 60, dict(hidden=6144 - 128), 32)])
def test_row_tiles_follow_tokens_per_expert_and_the_rounds_of_a_launch(workload, per, dims, rows):
    from dataclasses import replace
    spec = replace(C.workload(workload).spec, **dims)
    tokens = -(-per * spec.n_experts // spec.top_k)
    assert tokens * spec.top_k < (per + 1) * spec.n_experts
    assert _tiles(workload, tokens, **dims) == rows


def test_row_tiles_of_edge_calls():
    assert _tiles("c2_bf16_prefill", 1) == 1          # one token: no tiles
    assert _tiles("c2_bf16_prefill", 2) == 32
    assert _tiles("c2_bf16_prefill", 4096) == 128
    assert _tiles("c2_bf16_prefill", 4097) == 0       # more than one chunk holds
    assert _tiles("c2_bf16_prefill", 16, hidden=100) == 0
