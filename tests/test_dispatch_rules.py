"""Where the lines of rules lie that choose between kernels with the same results."""
import pytest


@pytest.fixture(scope="module")
def lib():
    from leone_amd.ops.library import library
    return library()


@pytest.mark.parametrize("longest,entries,heads,threads", [
    (1, 64, 16, 64), (2, 64, 16, 64), (64, 1, 4, 64),            # a wave has an entry's rows: no more threads than that
    (65, 1, 4, 256), (256, 8, 16, 256), (2000, 129, 32, 256),    # few trips, or many workgroups that share units
    (257, 1, 4, 1024), (2000, 16, 16, 1024), (257, 64, 16, 512), (2000, 128, 16, 512)])
def test_threads_of_the_exponential_gates(lib, longest, entries, heads, threads):
    assert lib.leone_exp_gates_threads(longest, entries, heads) == threads


@pytest.mark.parametrize("rows,heads,write_cache,runs", [(255, 100, 1, 0), (256, 14, 1, 1), (256, 13, 1, 0), (512, 4, 1, 0), (512, 8, 0, 0), (512, 9, 0, 1), (256, 17, 0, 0),
                                                         (256, 18, 0, 1), (2114, 24, 1, 1), (1 << 30, 24, 1, 1)])
def test_heads_of_wide_rows_in_runs(lib, rows, heads, write_cache, runs):
    assert lib.leone_heads_in_pairs(rows, heads, write_cache) == runs


@pytest.mark.parametrize("kind,each,n,runs", [("BF16", 1, 8 * 2048, 0), ("BF16", 1, 192 * 2048 - 8, 0), ("BF16", 1, 192 * 2048, 1), ("F32", 1, 96 * 2048 - 8, 0),
                                              ("F32", 1, 96 * 2048, 1), ("BF16", 0, 8, 1), ("F32", 1, 1 << 33, 1)])
def test_gates_in_runs(lib, kind, each, n, runs):
    from leone_amd import ops
    assert lib.leone_gates_in_runs(getattr(ops, kind), each, n) == runs


@pytest.mark.parametrize("experts,gated,n,k,one", [(8, 1, 2048, 4096, 1), (8, 0, 4096, 2048, 1), (16, 1, 1024, 2048, 1), (8, 1, 1856, 4096, 1), (8, 1, 1792, 4096, 0),
                                                   (8, 1, 2049, 4096, 0), (32, 1, 768, 2048, 0), (8, 1, 2048, 5120, 0), (4, 1, 2048, 4096, 0), (32, 1, 512, 4096, 0)])
def test_chunks_of_experts_matrices_on_their_way(lib, experts, gated, n, k, one):
    assert lib.leone_moe_one_chunk_ahead(experts, gated, n, k) == one


@pytest.mark.parametrize("m, n, k, kind, takes", [
    (17, 1024, 8192, "store", False), (48, 4096, 4096, "store", False), (49, 4096, 4096, "store", True), (33, 4096, 2048, "store", True),
    (33, 1024, 1024, "gated", True), (33, 2048, 2048, "gated", False), (33, 6144, 2048, "gated", True), (17, 24576, 4096, "gated", True), (33, 4096, 4096, "gated", False),
    (66, 14912, 5760, "store", False), (95, 19264, 5120, "store", False), (65, 32768, 4096, "store", True), (92, 6528, 5120, "store", True), (96, 24576, 4096, "gated", False),
    (96, 6144, 6144, "gated", True), (65, 16384, 4096, "gated", False), (128, 16384, 4096, "gated", True), (65, 15360, 2560, "store", False), (112, 15360, 2560, "store", True),
    (22, 18432, 3072, "gated", True), (17, 12288, 3072, "gated", False),                 # 192 workgroups of 96 and of 64 columns
    (17, 1024, 8192, "planes", True), (46, 9024, 3264, "planes", False), (128, 8192, 1024, "planes", True),
])
def test_which_products_of_up_to_128_rows_take_the_copy(m, n, k, kind, takes):
    """In one range of K few workgroups walk all of it, which the waves of ``gemm_rows`` share; large matrices are not read twice."""
    import torch

    from leone_amd import ops
    kind_of = torch.bfloat16 if kind == "gated" else torch.float32
    plan = ops._deep_sizes(m, n, k, kind == "planes", kind == "gated", kind_of, 256)
    assert (plan is not None) == takes and (plan is None or plan == ops.deep_plan(m, n, k, kind == "planes", kind == "gated"))


@pytest.mark.parametrize("experts,each,hidden,ff,gated,tile", [
    (32, 9, 2048, 768, True, 16), (32, 40, 2048, 768, True, 64), (32, 240, 2048, 768, True, 128), (8, 13, 4096, 2048, True, 0), (64, 60, 2048, 1408, True, 128),
    (4, 200, 512, 320, True, 64),                                           # tiles of 128 for less than half of the units
    (2, 31, 3520, 3968, True, 0), (8, 26, 2176, 1536, True, 0), (8, 34, 2688, 5696, True, 0), (8, 15, 5248, 3136, True, 0), (4, 31, 2944, 1216, True, 0), (4, 31, 1024, 1024, True, 64)])
def test_tiles_of_experts_products_from_their_copies(experts, each, hidden, ff, gated, tile):
    """Few workgroups that each walk a long inner size are slower than the kernels that read the matrices themselves (0)."""
    from leone_amd import ops
    assert ops._copied_tile(experts * each, experts, hidden, ff, gated, 256) == tile


@pytest.mark.parametrize("shape,carries", [("qwen3", False), ("zukinex", False), ("pamevik", True), ("fosulix", True), ("nogidra", True), ("reverax", True),
                                           ("sonulorn", True)])
def test_which_models_carry_memories(shape, carries):
    import torch

    from leone_amd import benchmark
    from leone_amd.architectures import config_from_dict, model_spec_for
    from leone_amd.parts.model import DecoderModel
    raw = dict(benchmark.QWEN3_8B, num_hidden_layers=2) if shape == "qwen3" else getattr(benchmark, shape + "_shape")(512, 4, 256, 256)
    model = DecoderModel(model_spec_for(config_from_dict(raw)), torch.bfloat16, torch.device("cpu"))
    assert model.carries_memories() == carries
    silent = DecoderModel.__new__(DecoderModel)
    silent.layers = [*model.layers, object()]              # a layer that does not say what it keeps
    assert silent.carries_memories()
