"""The fp4 form of the tiled scores: the same scores as the float16 form (bit for bit where the sums are exact), sums that
round, and operands of which only a part is exact in fp4."""

import pytest
import torch

from moespresso_amd import _lib

pytestmark = pytest.mark.gpu


def _operands(batch, heads, tokens, rows, dtype, seed=3):
    from moespresso_amd.runtime.deepseek_v4 import indexed_attention_kernel as iak
    from moespresso_amd.runtime.deepseek_v4 import indexer_score_kernel as isk

    gen = torch.Generator(device="cuda").manual_seed(seed)
    q = iak.indexer_q_qat_live(torch.randn((batch, heads, tokens, 128), device="cuda", generator=gen))
    comp = isk.indexer_qat_rows(torch.randn((batch, rows, 128), device="cuda", generator=gen))
    w = torch.randn((batch, tokens, heads), device="cuda", generator=gen)
    return q.to(dtype), w, comp.to(dtype)


def _both(q, w, comp, pos0, ratio=4):
    """(the operator's scores, the float16 form's scores)"""
    from moespresso_amd.runtime.deepseek_v4 import indexed_attention_kernel as iak

    got = iak.indexer_scores_tiled_live(q, w, comp, pos0=pos0, ratio=ratio)
    want = torch.empty_like(got)
    _lib.check(_lib.lib().mspr_indexer_scores_tiled_live(
        _lib.ptr(q), _lib.ptr(w), _lib.ptr(comp), _lib.DTYPE_CODE[q.dtype], q.shape[0], q.shape[1], q.shape[2],
        comp.shape[1], pos0, ratio, _lib.ptr(want), _lib.stream_ptr()), "float16 form")
    return got, want


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("batch,heads,tokens,rows,pos0,ratio", [
    (1, 64, 1, 1, 3, 4), (1, 64, 4, 31, 200, 4), (2, 64, 5, 33, 60, 4), (1, 64, 9, 63, 0, 0), (1, 64, 6, 64, 250, 4),
    (3, 64, 3, 65, 300, 4), (1, 40, 7, 130, 512, 4), (1, 1, 2, 97, 400, 4), (1, 64, 37, 2011, 7900, 4), (1, 64, 801, 1000, 0, 1)])
def test_qat_operands_give_the_float16_form_bit_for_bit(dtype, batch, heads, tokens, rows, pos0, ratio):
    got, want = _both(*_operands(batch, heads, tokens, rows, dtype), pos0, ratio)
    assert got.equal(want)
    assert ratio != 0 or bool(torch.isfinite(got).all())


# On both sides of the lines from which the fp4 form is taken (float32: more than 256 pieces of four tokens by 64 rows, and more
# than 64 rows; float16: 4096 pairs of a token and 64 rows, and 3072 and twice the packed blocks): ragged blocks of rows, tokens
# and heads, several sequences, the whole pool visible.
@pytest.mark.parametrize("dtype,batch,heads,tokens,rows,pos0,ratio", [
    (torch.float32, 1, 64, 4097, 33, 0, 4), (torch.float32, 2, 64, 1025, 64, 60, 4), (torch.float32, 1, 40, 1031, 130, 512, 4),
    (torch.float32, 3, 64, 46, 1000, 3800, 4), (torch.float32, 1, 1, 45, 3001, 11980, 4), (torch.float32, 1, 64, 6, 22011, 0, 0),
    (torch.float32, 1, 64, 2, 65535, 0, 0), (torch.float32, 1, 64, 2, 65536, 0, 0),
    (torch.float16, 1, 64, 4097, 129, 0, 4), (torch.float16, 2, 64, 1001, 255, 60, 4), (torch.float16, 1, 40, 3511, 130, 512, 4),
    (torch.float16, 3, 64, 150, 1024, 3800, 4), (torch.float16, 1, 1, 151, 2999, 11900, 4), (torch.float16, 1, 64, 22, 22011, 0, 0),
    (torch.float16, 1, 64, 18, 24999, 0, 0), (torch.float16, 1, 64, 18, 25000, 0, 0),
    (torch.float32, 1, 64, 64, 1024, 0, 0), (torch.float32, 1, 64, 65, 1024, 0, 0), (torch.float32, 1, 64, 64, 1025, 0, 0),
    (torch.float32, 1, 64, 1, 16384, 0, 0), (torch.float32, 1, 64, 1, 16385, 0, 0), (torch.float32, 2, 64, 515, 64, 0, 0),
    (torch.float32, 2, 64, 515, 65, 0, 0), (torch.float16, 1, 64, 256, 1024, 0, 0), (torch.float16, 1, 64, 257, 1024, 0, 0),
    (torch.float16, 1, 64, 256, 1025, 0, 0), (torch.float16, 2, 64, 130, 1024, 0, 0), (torch.float16, 1, 64, 1537, 200, 0, 0),
    (torch.float16, 1, 64, 1544, 200, 0, 0)])
def test_both_forms_agree_where_the_fp4_form_is_taken(dtype, batch, heads, tokens, rows, pos0, ratio):
    got, want = _both(*_operands(batch, heads, tokens, rows, dtype), pos0, ratio)
    assert got.equal(want)


@pytest.mark.parametrize("spoil", ["query", "pool", "tiny", "huge", "nan"])
def test_operands_outside_the_format_take_the_float16_form(spoil):
    q, w, comp = _operands(1, 64, 13, 200, torch.float32)
    if spoil == "query":
        q[0, 5, 6, 70] += 0.03125  # one token of the second workgroup
    elif spoil == "pool":
        comp[0, 199, 127] = 0.3
    elif spoil == "tiny":
        comp[0, 64, :32] *= 2.0 ** -20
    elif spoil == "huge":
        q[0, :, 2, 32:64] *= 2.0 ** 13
    else:
        comp[0, 3, 3] = float("nan")
    got, want = _both(q, w, comp, 900)
    assert torch.equal(torch.nan_to_num(got, nan=12345.0), torch.nan_to_num(want, nan=12345.0))


# (a block of 64 heads or pool rows is read on only if its first eight are of the format)
@pytest.mark.parametrize("operand,row", [("query", 0), ("query", 7), ("query", 8), ("query", 63), ("pool", 64 + 7), ("pool", 64 + 8),
                                         ("pool", 199), ("pool", 192)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_one_value_outside_the_format_anywhere_in_a_block(operand, row, dtype):
    from moespresso_amd.runtime.deepseek_v4 import indexed_attention_kernel as iak

    q, w, comp = _operands(1, 64, 2301, 200, dtype)
    if operand == "query":
        q[0, row, 633, 127] = 0.3
    else:
        comp[0, row, 127] = 0.3
    got, want = _both(q, w, comp, 900)
    assert got.equal(want)
    assert iak.indexer_scores_tiled_live(q, w, comp, pos0=900, qat_operands=False).equal(want)


@pytest.mark.parametrize("spoil", ["tiny", "huge", "nan"])
def test_groups_outside_the_scales_and_nan_among_many_scores(spoil):
    q, w, comp = _operands(1, 64, 701, 200, torch.float32)
    if spoil == "tiny":
        comp[0, 64, :32] *= 2.0 ** -20
    elif spoil == "huge":
        q[0, :, 2, 32:64] *= 2.0 ** 13
    else:
        comp[0, 103, 3] = float("nan")
    got, want = _both(q, w, comp, 900)
    assert torch.equal(torch.nan_to_num(got, nan=12345.0), torch.nan_to_num(want, nan=12345.0))


def _lattice_rows(rows, low, high, gen):
    """[rows, 128] of e2m1 lattice values, each group of 32 times a power of two with an exponent in [low, high]."""
    v = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], device="cuda")[torch.randint(0, 8, (rows, 128), device="cuda", generator=gen)]
    v *= torch.randint(0, 2, v.shape, device="cuda", generator=gen) * 2 - 1
    v[:, ::32] = 6.0                                 # (a group is stored by its largest magnitude)
    e = torch.randint(low, high + 1, (rows, 4), device="cuda", generator=gen)
    return v * torch.exp2(e.float()).repeat_interleave(32, dim=1)


@pytest.mark.parametrize("q_exp,comp_exp", [((0, 5), (-4, 0)), ((-13, -8), (9, 13))])
def test_group_exponents_within_nine_give_exact_sums(q_exp, comp_exp):
    gen = torch.Generator(device="cuda").manual_seed(4)
    q, comp = _lattice_rows(470, *q_exp, gen), _lattice_rows(300, *comp_exp, gen)
    got, want = _both(q.reshape(1, 1, 470, 128), torch.ones((1, 470, 1), device="cuda"), comp.reshape(1, 300, 128), 0, 0)
    assert got.equal(want)
    exact = torch.relu(q.double().cpu() @ comp.double().cpu().T)
    assert got[0].cpu().double().equal(exact)


def test_group_exponents_far_apart_round_in_float32():
    """One head of weight one, so that a score is a dot product. Either form adds its 128 products in at most eight
    instructions, each rounding its sum, at most the sum of magnitudes, to float32 (2^-23 allows a truncated sum)."""
    gen = torch.Generator(device="cuda").manual_seed(5)
    q, comp = _lattice_rows(300, -13, 13, gen), _lattice_rows(500, -13, 13, gen)
    got, f16 = _both(q.reshape(1, 1, 300, 128), torch.ones((1, 300, 1), device="cuda"), comp.reshape(1, 500, 128), 0, 0)
    assert not got.equal(f16)                        # (the fp4 form did the work)
    q, comp = q.double().cpu(), comp.double().cpu()
    exact, size = torch.relu(q @ comp.T), q.abs() @ comp.abs().T
    errors = [(x[0].cpu().double() - exact).abs() for x in (got, f16)]
    assert all(bool((e <= 8 * 2.0 ** -23 * size).all()) for e in errors)
    assert errors[0].norm() <= errors[1].norm()      # no less precise than the form it takes the place of


# The last sizes of the float16 form and the first of the fp4 form, told apart by how such sums round.
@pytest.mark.parametrize("dtype,tokens,rows,fp4", [
    (torch.float32, 64, 1024, False), (torch.float32, 65, 1024, True), (torch.float32, 64, 1025, True), (torch.float32, 2060, 64, False),
    (torch.float32, 2060, 65, True), (torch.float16, 256, 1024, False), (torch.float16, 257, 1024, True),
    (torch.float16, 1537, 200, False), (torch.float16, 1544, 200, True)])
def test_which_form_is_taken_on_either_side_of_its_line(dtype, tokens, rows, fp4):
    gen = torch.Generator(device="cuda").manual_seed(6)
    q, comp = _lattice_rows(tokens, -12, 12, gen).to(dtype), _lattice_rows(rows, -12, 12, gen).to(dtype)
    got, f16 = _both(q.reshape(1, 1, tokens, 128), torch.ones((1, tokens, 1), device="cuda"), comp.reshape(1, rows, 128), 0, 0)
    assert got.equal(f16) != fp4
