"""Which kernel of the hybrid library takes a call: the library's own rules, by sizes, strides and addresses."""
import pytest

from minivllm_amd.ops import hip_hybrid as hk

AT = 1 << 20                                           # an address of whole runs


@pytest.mark.parametrize("D,E,v_stride,shift,q_row,form", [
    # whole runs everywhere; whole key rows alone: the score products of the 16-bit instruction; neither
    (128, 128, 128, 0, 2048, 2), (128, 100, 100, 0, 2048, 1), (64, 20, 20, 0, 512, 1), (64, 64, 68, 0, 512, 1),
    (36, 64, 64, 0, 512, 0), (24, 20, 20, 0, 512, 0), (128, 100, 100, 2, 2048, 0), (128, 100, 100, 0, 2052, 0)])
def test_prompt_attention(D, E, v_stride, shift, q_row, form):
    a = (AT + shift, q_row, D, AT, AT, AT, 8, 1024, D, E, v_stride)
    assert hk._tiles_form(*a, 0) == form
    # float rows: the kernels of whole runs or the general one
    assert hk._tiles_form(*a, 2) == (2 if form == 2 else 0)
    # a value cache or an output off 16 bytes takes nothing from the score products
    if form == 2:
        assert hk._tiles_form(*a[:4], AT + 2, *a[5:], 0) == 1 and hk._tiles_form(*a[:5], AT + 2, *a[6:], 0) == 1


@pytest.mark.parametrize("H,G,D,E,taps,row,form", [
    (16, 8, 128, 128, 4, 6208, 2), (2, 1, 8, 8, 2, 32, 2), (2, 1, 2048, 8, 3, 4128, 2), (16, 8, 128, 128, 5, 6208, 0),
    # heads that are no whole runs in rows that are; no runs at all
    (16, 8, 100, 128, 4, 3680, 1), (16, 8, 36, 64, 2, 1632, 1), (8, 4, 2050, 8, 3, 16480, 1),
    (15, 15, 12, 12, 3, 572, 0), (3, 3, 12, 12, 3, 120, 0), (6, 3, 128, 128, 4, 1548, 0)])
def test_delta_preparation(H, G, D, E, taps, row, form):
    a = [AT, row, AT, AT, AT, AT, AT, taps, H, G, D, E]
    assert hk._prep_form(*a) == form
    for off in (2, 4, 5):                              # the taps' table and the unit vectors' address: the rows kernel only
        b = list(a)
        b[off] += 4
        assert hk._prep_form(*b) == (min(form, 1) if G * D % 8 == 0 else form)
    for off in (0, 3, 6):
        b = list(a)
        b[off] += 4
        assert hk._prep_form(*b) == 0


def test_heads_of_a_decode_workgroup():
    """No workgroup more than groups of four need, no head worked out twice that could be left out."""
    assert [hk._split_heads(r) for r in range(1, 13)] == [1, 2, 3, 4, 3, 3, 4, 4, 3, 4, 4, 4]


@pytest.mark.parametrize("batch,kv_heads,heads,longest,splits", [
    (64, 8, 16, 1024, 2), (64, 8, 16, 2048, 2), (32, 8, 16, 4096, 4), (1, 8, 16, 100, 1), (1, 8, 16, 8192, 16),
    # a long context in a batch that fills the card: spans of up to 2048 keys, eight workgroups per CU at most
    (64, 8, 16, 8192, 4), (128, 8, 16, 4096, 2), (128, 8, 16, 2048, 1), (256, 8, 16, 1 << 17, 1), (16, 8, 64, 1 << 17, 8),
    # an unknown context
    (64, 8, 16, 0, 2), (1, 8, 16, None, 8)])
def test_splits_of_a_decode_batch(batch, kv_heads, heads, longest, splits):
    assert hk.decode_splits(batch, kv_heads, heads, longest) == splits


@pytest.mark.parametrize("columns,keys,H,nseq,max_q,rows,form", [
    (128, 32, 8, 4, 32, 0, 41), (128, 33, 8, 4, 33, 0, 22), (128, 95, 8, 4, 95, 0, 22), (128, 96, 8, 4, 96, 0, 24),
    (192, 255, 8, 4, 128, 0, 22), (192, 256, 8, 4, 128, 0, 24), (256, 4096, 8, 4, 256, 0, 22),
    # 256 tiles of 64 queries, 264; 512, 520
    (192, 1023, 8, 4, 512, 0, 24), (192, 511, 8, 3, 704, 0, 22), (192, 512, 8, 3, 704, 0, 24), (192, 191, 8, 3, 704, 0, 41),
    (128, 191, 8, 3, 704, 0, 22), (256, 191, 8, 3, 704, 0, 41), (256, 192, 8, 3, 704, 0, 22), (192, 512, 8, 4, 1024, 0, 22),
    (192, 1024, 8, 4, 1024, 0, 24), (192, 383, 8, 5, 832, 0, 41), (192, 384, 8, 5, 832, 0, 42), (256, 383, 8, 5, 832, 0, 41),
    (256, 384, 8, 500, 832, 0, 42),
    # tiles of 128 queries: 384, 392; 512, 520; 640, 648
    (128, 384, 8, 16, 384, 0, 42), (128, 384, 8, 49, 128, 0, 41), (128, 512, 8, 64, 128, 0, 42), (128, 512, 8, 65, 128, 0, 41),
    (128, 1024, 8, 80, 128, 0, 42), (128, 1024, 8, 81, 128, 0, 41),
    # rows that are known: 8 * (4000 / 64 + 5) tiles at most
    (128, 1024, 8, 9, 1024, 4000, 42), (128, 1024, 8, 9, 1024, 0, 42), (128, 384, 8, 9, 1024, 4000, 42), (128, 384, 8, 9, 1024, 0, 41)])
def test_prompt_attention_form_of_float_rows(columns, keys, H, nseq, max_q, rows, form):
    assert hk._f32_form(columns, keys, H, nseq, max_q, rows) == form


@pytest.mark.parametrize("D,E,keys,workgroups,groups", [
    (128, 128, 384, 256, 2), (128, 128, 383, 256, 1), (128, 128, 4096, 257, 1), (256, 64, 384, 1, 2), (64, 256, 639, 1, 1),
    (64, 256, 640, 1, 2), (256, 128, 639, 1, 1), (256, 128, 640, 256, 2)])
def test_prompt_attention_groups(D, E, keys, workgroups, groups):
    assert hk._prompt_groups(D + E, E, keys, workgroups) == groups


@pytest.mark.parametrize("blocks,size,window,keep,chunk,walk", [
    (6, 64, 0, 0, 0, 384), (6, 64, 256, 0, 0, 383), (6, 64, 256, 4, 0, 384), (100, 64, 256, 4, 0, 387), (100, 64, 0, 0, 512, 639),
    (1 << 30, 1 << 20, 0, 0, 0, 1 << 30)])
def test_longest_walk(blocks, size, window, keep, chunk, walk):
    assert hk._longest_walk(blocks, size, window, keep, chunk) == walk


@pytest.mark.parametrize("B,H,D,E,one", [
    (64, 16, 128, 128, True), (255, 16, 128, 128, True), (256, 16, 128, 128, False), (127, 32, 128, 128, True),
    (128, 32, 128, 128, False), (512, 8, 256, 64, False), (256, 16, 64, 64, True), (257, 16, 64, 64, False),
    (1024, 4, 48, 40, True), (1025, 4, 48, 40, False)])
def test_next_tokens_of_the_delta_rule(B, H, D, E, one):
    """One kernel up to 256 MB of state and 4096 heads, the three calls beyond."""
    assert hk.delta_next_pays(B, H, D, E) is one


@pytest.mark.parametrize("T,H,R,prompts,few", [
    # rows of the caches and the weights: up to 2^18 of them times the rank, as the heads allow
    (512, 16, 512, True, True), (513, 16, 512, True, False), (4096, 8, 64, True, True), (4097, 8, 64, True, False),
    # ... times the heads: prompts up to 5 x 2^20, single next tokens up to 3 x 2^20
    (160, 64, 512, True, True), (161, 64, 512, True, False), (80, 128, 512, True, True), (1200, 64, 64, True, True),
    (96, 64, 512, False, True), (97, 64, 512, False, False), (48, 128, 512, False, True), (64, 128, 512, False, False),
    (256, 16, 512, False, True), (1, 128, 512, False, True)])
def test_few_rows_in_latents(T, H, R, prompts, few):
    assert hk.latent_rows_pay(T, H, R, prompts) is few


@pytest.mark.parametrize("B,H,D,E,each", [
    # walks of 32 columns: 32, 256, 512, 1024, 4096; (bfloat16, float) tokens a portion
    (1, 8, 128, 128, (32, 24)), (8, 8, 128, 128, (24, 16)), (8, 16, 128, 128, (16, 10)), (32, 8, 128, 128, (10, 10)),
    (128, 8, 128, 128, (8, 8)), (32, 16, 72, 264, (8, 8)),
    # up to 64 channels: 16, 256, 257, 1024, 1026, 4096
    (1, 8, 64, 64, (40, 40)), (16, 8, 64, 64, (40, 32)), (257, 1, 8, 8, (24, 32)), (64, 8, 64, 64, (24, 32)),
    (171, 3, 48, 40, (16, 32)), (256, 8, 64, 64, (16, 32))])
def test_matrix_lstm_portions_in_chunks(B, H, D, E, each):
    """As many tokens as make up for the portions, or one long portion among them; many small bfloat16 heads in one kernel."""
    walks = B * H * -(-E // 32)
    for dt in (0, 2):
        at = lambda T, longest, q=AT, row=8192, D=D: hk._mlstm_bytes(q, AT, AT, row, row, row, T, B, longest, H, D, E, dt)
        n = each[dt // 2]
        alone = 40 + walks // (64 if dt == 2 and D <= 64 else 200)
        assert at(n * B, n) and not at(n * B - 1, n - 1)
        if alone + B - 1 < n * B:
            assert at(alone + B - 1, alone) and not at(alone + B - 2, alone - 1)
        # an unknown length: as if it was all the rows beyond the first of each
        if B + 1024 < n * B:
            assert at(B + 1024, 0) and not at(B + 1023, 0)
        whole = dt == 0 and D <= 64 and walks > 256
        for T in (n * B, n * B + 640):
            assert at(T, n) == at(T, -1) == (256 if whole else (T // 64 + B) * H * 1024) <= hk.mlstm_scan_workspace(T, B, H, D, E)
        assert at(B, -1) and not at(n * B, n, AT + 2) and not at(n * B, n, AT, 8190) and not at(n * B, n, D=136)
