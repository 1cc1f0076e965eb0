"""Which decode steps over latents go to the three launches built for them: the sizes, and heads, sequences and contexts on both
sides of the line, at the points where both ways were timed (no GPU)."""
import pytest
import torch


@pytest.mark.parametrize("rank,heads,n,context,three", [
    (512, 16, 1, 60, True), (512, 16, 8, 700, True), (512, 16, 64, 16000, True), (512, 16, 128, 16000, False), (512, 16, 1, 64000, True),
    (512, 17, 8, 700, True), (512, 32, 128, 1000, True), (512, 32, 64, 4000, False), (512, 64, 64, 1000, True),
    (512, 64, 32, 4000, False), (512, 64, 128, 1000, False), (512, 128, 8, 4000, True), (512, 128, 64, 1000, False),
    (512, 128, 8, 16000, False), (512, 128, 128, 180, True), (256, 16, 128, 1000, True), (256, 16, 64, 16000, False),
    (256, 40, 64, 1000, False), (256, 128, 128, 180, True), (128, 16, 32, 4000, True), (128, 16, 64, 4000, False)])
def test_heads_sequences_and_contexts(rank, heads, n, context, three):
    from pytorch_transformers_amd import ops

    if not ops.LATENT_DECODE:
        pytest.skip("switched off by PTA_LATENT_DECODE=0")
    x = torch.empty((n, 1), dtype=torch.bfloat16)
    assert ops.latent_decode_ok(x, heads, 128, 64, rank, 128, context) is three
    # a captured step, padded to its bucket and sized for its bound, takes the way of the same step run directly
    bucket = n if n <= 8 else (n + 7) // 8 * 8
    from pytorch_transformers_amd import tuning

    assert ops.latent_decode_ok(torch.empty((bucket, 1), dtype=torch.bfloat16), heads, 128, 64, rank, 128, tuning.context_bound(context)) is three
    assert ops.latent_ranges(n, heads, context) == ops.latent_ranges(bucket, heads, tuning.context_bound(context))


@pytest.mark.parametrize("n,heads,context", [(1, 16, 1), (1, 16, 16000), (1, 16, 1_000_000), (3, 40, 5000), (64, 16, 700), (300, 128, 70)])
def test_ranges_cover_the_context(n, heads, context):
    from pytorch_transformers_amd import ops

    size, ranges = ops.latent_ranges(n, heads, context)
    assert size % 64 == 0 and 1 <= ranges <= 1024 and size * ranges >= context > 0
    assert (ranges - 1) * size < max(192, (context + 1023) // 1024 * 1024)


def test_the_turned_matrix_is_kept_where_it_is_read():
    from pytorch_transformers_amd import ops
    from pytorch_transformers_amd.parts import LatentAttentionMixer, RotaryPositions

    def turned(dtype, rank):
        m = LatentAttentionMixer("m", 64, 2, 32, 32, 16, rank, 0.1, 1e-5, RotaryPositions(32, 10000.0))
        m.load_all({s.name: torch.zeros(s.shape, dtype=dtype) for p in [m, *m.children()] for s in p.tensor_specs()})
        m.after_load()
        return m.k_turned

    assert turned(torch.float32, 64) is None and turned(torch.bfloat16, 40) is None
    kept = turned(torch.bfloat16, 64)
    assert (kept is None) == (not ops.LATENT_DECODE) and (kept is None or kept.shape == (2, 64, 32))
