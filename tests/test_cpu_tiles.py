"""The GPU tests of the fp32 tiles run every tile: their shapes against the
choices that the launches make (no GPU)."""
import test_gpu_fp32_batch as batch
import test_gpu_matmul_tiles as matmul
import tile_choice as choice


def test_matmul_shapes_take_every_form():
    assert {choice.matmul_form(*s) for s in matmul.SHAPES} == choice.MATMUL_FORMS


def layer_forms(shape, tokens):
    heads, kv_heads, head_dim, ffn, _ = shape
    dim, kv = heads * head_dim, kv_heads * head_dim
    for epilogue, k, n in (("qkv", dim, dim + 2 * kv), ("add", dim, dim), ("swiglu", dim, 2 * ffn),
                           ("add", ffn, dim)):
        yield (epilogue, *choice.fgemm_form(epilogue, tokens, k, n))


def test_fp32_prompts_take_every_projection_form():
    have = set()
    for shape, tokens in batch.WIDE.values():
        for t in tokens:
            have.update(layer_forms(shape, t))
    for shape in batch.SHAPES.values():
        for t in (1, 2, 15, 16, 17, 64, 65, 300):
            have.update(layer_forms(shape, t))
    # every tile of the table in every projection, and the forms of up to 16 rows
    tiles = {(ti, tj, 8 if (ti, tj) == (1, 2) else 4, 1)
             for ti, tj, _ in choice.table("fmodel.hip", "template <int EPI> void launch_fgemm")}
    want = {(e, *t) for e in ("qkv", "add", "swiglu") for t in tiles}
    want |= {(e, 1, 4, 8, 1) for e in ("qkv", "swiglu")}
    want |= {(e, 1, 2, 16, 1) for e in ("qkv", "add", "swiglu")}
    want |= {("add", 1, 1, 16, 1)} | {("add", 1, 2, 8, runs) for runs in (2, 3, 4)}
    assert have == want, (have - want, want - have)
