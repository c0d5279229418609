"""Which kernel a product runs on (no GPU needed): the rules that share launches out between the decode, short-run and chunk kernels
have to agree with one another and with the overrides."""
import importlib
import random

import pytest

KINDS = ["int8", "nf4"]
SHAPES = {"int8": ([4096] * 4, 4096, 4), "nf4": ([2048] * 4, 2048, 3)}  # products that the short-run kernel takes from the decode kernels


@pytest.mark.parametrize("kind", KINDS)
def test_route_of_a_refused_product(wrq, kind):
    with pytest.raises(ValueError, match="multiple of 4"):
        wrq.debug_route(kind, 1022, 1024, 3)


@pytest.mark.parametrize("kind", KINDS)
def test_decode_runs_leave_for_the_short_run_kernel_only(wrq, kind):
    # what that kernel does not take has to stay on the decode kernels, not to end on the chunk kernel
    rows, K, T = SHAPES[kind]
    assert isinstance(wrq.debug_route(kind, rows, K, T), tuple)
    stride = (1 << 30) // (T - 1) + 8 & ~7  # a token's row more than 2 GiB behind the first one's: beyond its 32-bit offsets
    assert wrq.debug_route(kind, rows, K, T, x_token_stride=stride) == "decode"
    assert wrq.debug_route(kind, rows, K, T, x_token_stride=stride // 2 & ~7) != "decode"
    for K in (1 << 24, (1 << 24) + 1024, 0):
        for T in (1, 2, 3, 4):
            for rows in (4, 4096):
                assert wrq.debug_route(kind, rows, K, T) != "chunk" or (kind, T) == ("nf4", 4), (rows, K, T)
    rng = random.Random(5)
    for _ in range(2000):  # nf4 runs of 4 tokens are the matrix cores' in any case
        rows, K, T = [4 * rng.randint(1, int(2 ** rng.uniform(0, 14))) for _ in range(rng.randint(1, 8))], 128 * rng.randint(1, int(2 ** rng.uniform(0, 8))), rng.randint(2, 4)
        assert wrq.debug_route(kind, rows, K, T) != "chunk" or (kind, T) == ("nf4", 4), (rows, K, T)
    assert wrq.debug_route("int8", 4096, (1 << 24) + 1024, 4) == "decode"
    assert wrq.debug_route(kind, 4096, 0, 5) == "decode"


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("key,value", [("gemm_ntile", 1), ("gemm_mrt", 2), ("gemm_kg", 2), ("gemm_ksplit", 1), ("gemm_short", 0)])
def test_pinned_chunk_tiles_leave_decode_runs_alone(wrq, overrides, kind, key, value):
    rows, K, T = SHAPES[kind]
    assert isinstance(wrq.debug_route(kind, rows, K, 16), tuple)
    overrides(**{key: value})
    assert wrq.debug_route(kind, rows, K, T) == "decode"
    assert wrq.debug_route(kind, rows, K, 16) == "chunk"


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("key,value", [("gemv_oneshot", 1), ("gemv_rows", 8), ("gemv_nt", 128), ("gemv_sl", 1), ("gemv_grid", 256), ("gemv_waverows", 1), ("gemv_rows_tokens", 0)])
def test_pinned_decode_kernels_keep_their_runs(wrq, overrides, kind, key, value):
    rows, K, T = SHAPES[kind]
    assert isinstance(wrq.debug_route(kind, rows, K, T), tuple)
    overrides(**{key: value})
    assert wrq.debug_route(kind, rows, K, T) == "decode"
    assert isinstance(wrq.debug_route(kind, rows, K, 16), tuple)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("key", ["gemm_table", "gemv_table"])
def test_leaving_a_table_out_moves_no_product(wrq, overrides, kind, key):
    rows, K, T = SHAPES[kind]
    want = [wrq.debug_route(kind, rows, K, t) for t in (T, 16)]
    overrides(**{key: 0})
    assert [wrq.debug_route(kind, rows, K, t) for t in (T, 16)] == want


@pytest.mark.parametrize("kind,rows,K,T", [("int8", 65536, 4096, 8), ("int8", 65536, 4096, 16)])
def test_products_of_many_rows_keep_their_measured_tiles(wrq, kind, rows, K, T):
    # beyond the rows that the short-run kernel takes short runs are the chunk kernel's; its measured tiles beat its rules there (55.2 against 61.6 us at 8 tokens)
    from test_tuned_table import rows_of_table

    tune = importlib.import_module("web-rwkv_amd.tune_gemm")
    assert wrq.debug_route(kind, rows, K, T) == "chunk"
    bucket = next(i for i, t in enumerate(tune.T_GRID) if t >= T)
    assert any(cells[bucket] for q, r, k, cells in rows_of_table() if (q, r, k) == (KINDS.index(kind), rows, K))


@pytest.mark.parametrize("kind", KINDS)
def test_every_tile_of_the_short_run_kernel_has_a_test(wrq, overrides, kind):
    # the GPU tests compare that kernel with the chunk kernel on launches whose tile the rules choose
    import test_gpu_parity as gpu_tests

    built = {(1, 8, 8, 2)} | {(m, t, 8, 1) for m in (1, 2, 3, 4) for t in (8, 16, 24, 32)} | {(3, 24, 4, 1), (3, 32, 4, 1), (1, 48, 8, 1), (2, 48, 8, 1), (3, 48, 4, 1), (4, 48, 4, 1)}
    built |= {(4, 64, 4, 1)} if kind == "int8" else set()
    overrides(vec_chunk_min_t=2)
    launches = [(g, T) for g in gpu_tests.SHORT_GROUPS[kind] for T in gpu_tests.SHORT_T] + [(gpu_tests.SHORT_ROUNDS, T) for T in gpu_tests.SHORT_ROUNDS_T]
    launches += [(g, T) for g in gpu_tests.SHORT_BLOCKS for T in gpu_tests.SHORT_BLOCKS_T]
    seen = {wrq.debug_route(kind, [R for _, R in g], g[0][0], T) for g, T in launches} - {"chunk"}
    assert seen == built, (built - seen, seen - built)


@pytest.mark.parametrize("kind,rows,K,T,route", [
    # (slower there / faster there, as measured against the kernels that took these launches before)
    ("nf4", 1024, 4096, 3, "decode"), ("nf4", 1024, 5120, 3, "decode"), ("nf4", 1280, 4096, 3, "short"), ("nf4", 1024, 2560, 3, "short"),
    ("int8", 2048, 10240, 16, "chunk"), ("int8", 2048, 14336, 12, "chunk"), ("int8", 2048, 8192, 16, "short"), ("int8", 2560, 14336, 16, "short"),
    ("nf4", 2048, 14336, 16, "chunk"), ("nf4", 2048, 12288, 16, "short"), ("int8", 4096, 17920, 20, "chunk"), ("int8", 4096, 14336, 20, "short"), ("int8", 11260, 15488, 18, "short"),
    ("int8", 1024, 4096, 32, "chunk"), ("int8", 1280, 4096, 32, "short"), ("int8", 768, 4096, 28, "short"), ("nf4", 1024, 4096, 32, "short"),
    ("nf4", 4096, 16384, 32, "chunk"), ("nf4", 4096, 14336, 32, "short"), ("nf4", 5120, 17920, 32, "short"),
    ("nf4", 16384, 128, 48, "chunk"), ("int8", 16384, 128, 48, "chunk"), ("nf4", 5120, 128, 128, "chunk"), ("int8", 2560, 128, 256, "chunk"), ("nf4", 1024, 128, 128, "short"),
    ("int8", 4096, 8960, 128, "chunk"), ("int8", 4096, 10240, 112, "chunk"), ("int8", 2560, 10240, 128, "chunk"), ("int8", 2048, 10240, 224, "chunk"),
    ("int8", 2048, 8960, 256, "chunk"), ("int8", 2048, 8960, 192, "short"), ("int8", 2560, 8960, 128, "short"), ("int8", 5120, 10240, 96, "short"), ("int8", 3072, 10240, 160, "short"), ("int8", 4096, 8192, 128, "short"),
    ("nf4", 8192, 14336, 64, "chunk"), ("nf4", 4096, 10240, 128, "chunk"), ("nf4", 8192, 8192, 64, "short"), ("nf4", 8192, 14336, 48, "short"), ("nf4", 5120, 17920, 96, "short"),
    ("int8", 5120, 5120, 192, "chunk"), ("int8", 3072, 5120, 256, "chunk"), ("int8", 5120, 4096, 192, "short"), ("int8", 6144, 5120, 128, "short")])
def test_short_run_rules_end_where_the_other_kernels_are_faster(wrq, kind, rows, K, T, route):
    got = wrq.debug_route(kind, rows, K, T, mat=wrq.turbo(T))
    assert (got if isinstance(got, str) else "short") == route, got
