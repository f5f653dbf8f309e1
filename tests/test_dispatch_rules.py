"""The rules that choose between kernels, at calls where both sides were measured (no GPU needed)."""
import pytest

from vllm_distributed_amd.ops import hip


@pytest.mark.parametrize("kind,rows,seqs,longest,heads,dim,vdim,chunked", [
    # decoded rows, whatever their number; prompts of unknown lengths; heads the kernels are not built for
    (hip.DELTA_CHANNEL, 256, 256, 1, 16, 128, 128, False), (hip.LINEAR_HEAD, 1, 1, 1, 16, 128, 128, False),
    (hip.DELTA_HEAD, 256, 256, 0, 16, 128, 128, False), (hip.DELTA_HEAD, 2000, 2, 0, 16, 128, 128, True),
    (hip.LINEAR_CHANNEL, 8000, 1, 8000, 16, 129, 128, False), (hip.STATE_SPACE, 8000, 1, 8000, 16, 192, 64, False),
    # long prompts (chunked, row by row in us): 423 / 974, 260 / 597, 263 / 705, 223 / 831, 79 / 297, 61 / 87
    (hip.DELTA_CHANNEL, 8017, 5, 2000, 16, 128, 128, True), (hip.LINEAR_CHANNEL, 8017, 5, 2000, 16, 128, 128, True),
    (hip.LINEAR_HEAD, 8017, 5, 2000, 16, 128, 128, True), (hip.STATE_SPACE, 8017, 5, 2000, 16, 128, 128, True),
    (hip.DELTA_CHANNEL, 700, 1, 700, 16, 128, 128, True), (hip.DELTA_CHANNEL, 210, 2, 120, 32, 128, 128, True),
    # one short prompt: 34 / 38, of many heads 46 / 93
    (hip.DELTA_CHANNEL, 60, 1, 60, 8, 128, 128, True), (hip.DELTA_CHANNEL, 97, 1, 97, 64, 128, 128, True),
    # small heads, where a chunk costs more than its share of the products: 109 / 91, 101 / 72, 151 / 110
    (hip.LINEAR_HEAD, 960, 63, 300, 32, 16, 16, False), (hip.LINEAR_CHANNEL, 960, 63, 300, 32, 16, 16, False),
    (hip.DELTA_CHANNEL, 8990, 58, 155, 16, 16, 16, False)])
def test_chunked_recurrences_run_where_they_are_faster(kind, rows, seqs, longest, heads, dim, vdim, chunked):
    assert hip.chunk_scan_profitable(kind, rows, seqs, longest, heads, dim, vdim) is chunked


@pytest.mark.parametrize("kind,rows,seqs,longest,heads,dim,vdim,columns", [
    # prompts alike, and one longer than the others (32 / 16 columns, us): 128 / 160, 119 / 147; 176 / 145, 65 / 56, 161 / 134, 75 / 74
    (hip.DELTA_HEAD, 7000, 5, 1400, 8, 128, 128, 32), (hip.DELTA_HEAD, 7000, 6, 1167, 8, 128, 128, 32),
    (hip.DELTA_HEAD, 7000, 5, 2420, 8, 128, 128, 16), (hip.DELTA_HEAD, 1785, 5, 668, 8, 128, 128, 16),
    (hip.DELTA_HEAD, 7000, 6, 2065, 8, 128, 128, 16), (hip.DELTA_HEAD, 6038, 3, 2884, 16, 128, 128, 16),
    # 118 / 136, 292 / 340, 220 / 242; one prompt 284 / 350; a prompt beside decoded rows is by itself
    (hip.DELTA_HEAD, 7000, 7, 1200, 8, 128, 128, 32), (hip.DELTA_CHANNEL, 7000, 3, 2515, 16, 128, 128, 32),
    (hip.DELTA_CHANNEL, 8017, 5, 2000, 16, 128, 128, 32), (hip.DELTA_CHANNEL, 8000, 1, 8000, 32, 128, 128, 16),
    (hip.DELTA_CHANNEL, 2100, 101, 2000, 16, 128, 128, 16),
    # the longest is not known: as if all were alike
    (hip.DELTA_HEAD, 7000, 5, 0, 8, 128, 128, 32), (hip.DELTA_HEAD, 7000, 4, 0, 8, 128, 128, 16),
    # 64 keys; kinds without a delta rule
    (hip.DELTA_HEAD, 4000, 2, 2000, 32, 64, 128, 16), (hip.DELTA_HEAD, 4000, 4, 1000, 32, 64, 128, 32),
    (hip.LINEAR_HEAD, 4000, 4, 3000, 16, 128, 128, 32), (hip.STATE_SPACE, 4000, 3, 3000, 16, 128, 128, 16)])
def test_columns_of_the_chunked_walk(kind, rows, seqs, longest, heads, dim, vdim, columns):
    assert hip.chunk_columns(kind, rows, seqs, longest, heads, dim, vdim) == columns


@pytest.mark.parametrize("kind,rows,seqs,longest,heads,dim,vdim,least,most", [
    # decoded rows, heads and states the kernels are not built for
    (hip.LINEAR_CHANNEL, 256, 256, 1, 16, 128, 128, -1, -1), (hip.STATE_SPACE, 8000, 1, 8000, 16, 192, 128, -1, -1),
    (hip.LINEAR_HEAD, 8000, 1, 8000, 16, 128, 512, -1, -1),
    # long prompts, cut (chunked, segments in us): 205 / 149, 237 / 87, 113 / 56
    (hip.LINEAR_CHANNEL, 6007, 3, 2464, 16, 128, 128, 384, 512), (hip.STATE_SPACE, 7000, 1, 7000, 8, 128, 128, 128, 320),
    (hip.LINEAR_CHANNEL, 3000, 1, 3000, 8, 128, 128, 96, 160),
    # many short ones, whole: 108 / 75, 64 / 50, 85 / 53
    (hip.STATE_SPACE, 4000, 20, 400, 32, 64, 64, 0, 0), (hip.LINEAR_CHANNEL, 2512, 22, 195, 8, 128, 128, 0, 0),
    (hip.LINEAR_HEAD, 1017, 22, 94, 16, 128, 128, 0, 0),
    # the same against the walk, where chunks are further behind: 194 / 119, 298 / 214, 131 / 80, 97 / 45
    (hip.LINEAR_CHANNEL, 6000, 24, 250, 16, 128, 128, 0, 0), (hip.LINEAR_HEAD, 8964, 54, 166, 16, 128, 128, 0, 0),
    (hip.STATE_SPACE, 960, 63, 300, 32, 64, 64, 0, 0), (hip.LINEAR_CHANNEL, 1196, 11, 173, 16, 96, 96, 0, 0),
    # one round of segments; where a second one would be nearly empty chunked / segments 80 / 107, 72 / 88, 104 / 121
    (hip.LINEAR_HEAD, 6007, 3, 2434, 16, 128, 128, 384, 416), (hip.LINEAR_CHANNEL, 6007, 3, 2434, 16, 128, 128, 384, 416),
    (hip.LINEAR_HEAD, 6524, 13, 899, 16, 64, 64, -1, -1), (hip.LINEAR_HEAD, 5247, 10, 909, 16, 64, 64, -1, -1),
    (hip.LINEAR_HEAD, 1931, 1, 1931, 32, 128, 128, -1, -1),
    # many heads beside short rows: walk / segments 26 / 34
    (hip.LINEAR_CHANNEL, 710, 23, 50, 64, 32, 64, -1, -1),
    # few short ones, whose chains of 32 rows would be longer: 23 / 36, 32 / 44, 26 / 34
    (hip.LINEAR_HEAD, 215, 1, 215, 16, 64, 128, -1, -1), (hip.LINEAR_CHANNEL, 230, 1, 230, 32, 128, 128, -1, -1),
    (hip.STATE_SPACE, 668, 2, 374, 16, 64, 64, -1, -1)])
def test_segments_run_where_they_are_faster(kind, rows, seqs, longest, heads, dim, vdim, least, most):
    cut = hip.segment_rows(kind, rows, seqs, longest, heads, dim, vdim)
    assert least <= cut <= most and (cut <= 0 or cut % 32 == 0)


@pytest.mark.parametrize("cut,seqs,heads,vdim,goes", [(0, 1 << 20, 7, 8, True), (0, 1 << 20, 8, 8, False), (0, 1 << 19, 8, 136, False),
                                                      (96, 1, 65535, 16, True), (96, 1, 65536, 16, False)])
def test_segments_leave_what_a_launch_cannot_hold_to_other_kernels(monkeypatch, cut, seqs, heads, vdim, goes):
    import torch
    handed = []

    class Lib:
        @staticmethod
        def vdamd_segment_scan_floats(*sizes):
            return 1

        @staticmethod
        def vdamd_segment_scan(*args):
            handed.append(args)
            return 0
    monkeypatch.setattr(hip, "_LIB", Lib)
    monkeypatch.setattr(hip, "_stream", lambda: None)
    monkeypatch.setattr(hip, "segment_rows", lambda *sizes: cut)
    x, lens = torch.empty(1, heads * (16 + vdim)), torch.empty(seqs, dtype=torch.int32)
    out = hip._segment_scan(hip.LINEAR_HEAD, x, 0, heads * 8, heads * 16, None, None, None, x, None, heads, heads, 8, vdim, x, lens, lens,
                            lens, False, 1.0, 100)
    assert (out is not None) is goes is bool(handed)


@pytest.mark.parametrize("batch,heads,keys,captured,splits", [
    # (whole against split in us) 13.5 / 18 from Python; in a graph 12.5 / 8.5 and 9.3 / 9.0
    (1, 8, 800, False, 1), (1, 8, 800, True, 12), (8, 8, 520, True, 1), (1, 8, 512, True, 1), (1, 8, 1, False, 1),
    # a workgroup for most CUs: 18 / 20 and 20 / 22 in three; 22.5 / 25.9 in two; enough keys: 354 / 311
    (24, 8, 800, True, 1), (31, 8, 800, True, 1), (24, 8, 1000, False, 1), (32, 8, 1000, True, 1), (32, 8, 9000, False, 2),
    # 512 workgroups rather than more than that: 5 and 6 of 96 over 1000 keys 14.5 and 16
    (12, 8, 1000, True, 5), (20, 8, 1400, True, 3), (20, 8, 4000, False, 4), (16, 8, 3000, False, 4), (64, 8, 4000, True, 1), (1, 1, 100000, True, 64)])
def test_decode_splits(monkeypatch, batch, heads, keys, captured, splits):
    monkeypatch.setattr(hip, "MAX_SPLITS", 64, raising=False)
    assert hip.choose_num_splits(batch, heads, keys, captured) == splits
    # the workspace of a captured step serves every call of its size
    assert hip.decode_workspace_floats(batch, heads, 128, heads, keys) >= batch * splits * heads * 130


@pytest.mark.parametrize("tokens,heads,keys,by_token,seqs,rows_ok,captured,plan", [
    # decoded rows from Python: one launch up to 383 keys (13.6 / 20); in a graph split (12.7 / 10.6)
    (1, 16, 200, False, 1, True, False, (3, 1)), (1, 16, 200, False, 1, True, True, (3, 3)),
    (1, 16, 200, False, 1, False, False, (0, 1)), (1, 16, 4000, False, 1, True, False, (3, 62)),
    # no more workgroups than run at once: 26.8 / 32.6, 93 / 117, 23.7 / 32.5, whole rows 14.5 / 19.7 and 24.7 / 32.8
    (100, 16, 700, False, 100, True, True, (3, 5)), (160, 16, 3000, False, 160, True, True, (3, 3)),
    (130, 16, 400, False, 130, True, True, (3, 3)), (15, 128, 200, False, 15, True, True, (3, 1)),
    (256, 16, 400, False, 256, True, True, (3, 1)), (128, 16, 3100, False, 128, True, True, (3, 4)),
    # many heads by one, whatever the number of rows (four head tiles a workgroup, one): 167 / 101, 139 / 112, 346 / 288
    (69, 128, 780, False, 69, True, True, (3, 1)), (128, 128, 600, False, 128, True, True, (3, 1)),
    (256, 64, 1500, False, 256, True, True, (3, 1)), (20, 128, 3000, False, 20, True, True, (3, 3)),
    # prompts and verified rows over key rows (both caches, key rows): 47 / 31, 62 / 26, 231 / 133, 31 / 21, 56 / 24, 58 / 22, 50 / 32,
    # 42 / 30; from Python whole up to 383 keys (whole, split): 17.0 / 21.2; in a graph split: 17.4 / 12.8
    (200, 16, 700, True, 1, True, False, (3, 2)), (600, 16, 300, True, 2, True, False, (3, 1)),
    (1000, 16, 1500, True, 1, True, False, (3, 1)), (8, 16, 2000, True, 1, True, False, (3, 31)),
    (4, 16, 16000, True, 1, True, False, (3, 64)), (64, 16, 1000, True, 16, True, True, (3, 8)),
    (32, 128, 600, True, 1, True, False, (3, 2)), (8, 128, 2000, True, 1, True, False, (3, 8)),
    (32, 16, 300, True, 1, True, False, (3, 1)), (32, 16, 300, True, 1, True, True, (3, 4)),
    # caches whose key rows cannot be read.  Four head tiles a workgroup: 54 / 72, 118 / 149
    (40, 128, 500, False, 40, False, True, (2, 3)), (100, 128, 700, False, 100, False, True, (2, 1)),
    # prompts: 47 / 66, 65 / 92, rows of different lengths in two 227 / 269 and 102 / 116; 3 tokens of 16 sequences 50 / 56
    (200, 16, 700, True, 1, False, False, (1, 5)), (192, 32, 564, True, 3, False, False, (1, 2)),
    (1000, 16, 1000, True, 2, False, False, (1, 2)), (600, 16, 300, True, 2, False, False, (1, 2)),
    (700, 16, 700, True, 1, False, False, (1, 2)), (1500, 16, 1500, True, 1, False, False, (1, 1)),
    (48, 16, 1500, True, 16, False, True, (1, 9)), (32, 16, 300, True, 1, False, False, (1, 4))])
def test_latent_plan(tokens, heads, keys, by_token, seqs, rows_ok, captured, plan):
    assert hip.mla_plan(tokens, heads, keys, by_token, seqs, rows_ok, None, captured) == plan


@pytest.mark.parametrize("tokens,heads,keys,splits", [
    # whole / in two, us: 29 / 44, 30 / 49, 60 tokens behind 300 25 / 42, 31 / 43; in two / four 43 / 48; in one / three 42 / 34; 68 / 65
    (50, 128, 400, 1), (64, 128, 400, 1), (60, 128, 560, 1), (100, 64, 500, 1), (32, 128, 800, 2), (20, 128, 600, 3), (50, 128, 1500, 2),
    (100, 128, 4000, 1)])
def test_latent_splits_of_four_tiles_a_workgroup(tokens, heads, keys, splits):
    assert hip.mla_plan(tokens, heads, keys, False, tokens, True, 4, False) == (4, splits)


@pytest.mark.parametrize("rows_ok", [True, False])
def test_latent_attention_takes_the_plan(rows_ok, monkeypatch):
    """What ``mla_plan`` answers is what the kernels are handed; there is no rule beside it."""
    import torch
    handed = []

    class Lib:
        @staticmethod
        def vdamd_mla_attention(*args):
            handed.append(args[18:20])                 # splits, mode
            return 0
    monkeypatch.setattr(hip, "_LIB", Lib)
    monkeypatch.setattr(hip, "_stream", lambda: None)
    monkeypatch.setattr(hip, "mla_supported", lambda *shape: True)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    block = 32 if rows_ok else 16
    kc = torch.zeros(128 // block, 1, block, 320, dtype=torch.bfloat16)
    vc = torch.zeros(128 // block, 1, 16, block // 8, 16, 8, dtype=torch.bfloat16)
    for tokens, heads, by_token in ((9, 16, True), (40, 64, False), (2, 16, False)):
        table = torch.zeros(1 if by_token else tokens, 128 // block, dtype=torch.int32)
        hip.mla_attention(torch.zeros(tokens, heads, 320, dtype=torch.bfloat16), kc, vc, table,
                          torch.zeros(tokens, dtype=torch.int32) if by_token else None,
                          torch.full((tokens,), 100, dtype=torch.int32), 0.1, 100)
        mode, splits = hip.mla_plan(tokens, heads, 100, by_token, table.shape[0], rows_ok, None, False)
        assert handed[-1] == (splits, mode) and (mode == 3) is rows_ok


@pytest.mark.parametrize("tokens,heads,keys,captured,shared", [
    # single / shared, us: 29 / 26, 62 / 43, 39 / 36, 49 / 38, 172 / 115; 20 / 26, 31 / 34, 34 / 37; too few tiles; in a graph (27 / 22)
    (50, 128, 400, False, True), (20, 128, 1500, False, True), (5, 128, 4000, False, True), (12, 64, 4000, False, True),
    (100, 80, 3000, False, True), (1, 128, 3000, False, False), (8, 128, 1500, False, False), (8, 64, 4000, False, False),
    (4000, 48, 4000, False, False), (100, 128, 9000, True, True), (64, 128, 9000, True, False), (100, 128, 100, True, False)])
def test_latent_heads_shared(tokens, heads, keys, captured, shared, monkeypatch):
    """The rule, and that it decides where no kernel was asked for, weights precise or not; a kernel that was asked for is the one that
    runs."""
    import torch
    assert hip.mla_heads_shared(tokens, heads, keys, captured) is shared
    handed = []

    class Lib:
        @staticmethod
        def vdamd_mla_attention(*args):
            handed.append(args[18:20])                 # splits, mode
            return 0
    monkeypatch.setattr(hip, "_LIB", Lib)
    monkeypatch.setattr(hip, "_stream", lambda: None)
    monkeypatch.setattr(hip, "mla_supported", lambda *shape: True)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: captured)
    kc, vc = torch.zeros(4, 1, 32, 320, dtype=torch.bfloat16), torch.zeros(4, 1, 16, 4, 16, 8, dtype=torch.bfloat16)
    row = lambda n: torch.zeros(1, heads, n, dtype=torch.bfloat16).expand(tokens, heads, n)
    q, out, table = row(320), row(256), torch.zeros(tokens, 4, dtype=torch.int32)
    for mode, precise in ((None, False), (None, True), (3, False), (3, True), (4, False), (2, False), (0, False)):
        hip.mla_attention(q, kc, vc, table, None, torch.ones(tokens, dtype=torch.int32), 0.1, keys, out=out, mode=mode, precise=precise)
        assert handed[-1][1] == (mode if mode is not None else 4 if shared and not precise else 3)


@pytest.mark.parametrize("tokens,heads,keys,prompts,shared", [
    # single / shared, us: 28 / 33, 47 / 53, 44 / 48, 153 / 159; 61 / 50, 37 / 33, 162 / 134; windows
    (200, 96, 200, 1, False), (400, 128, 100, 4, False), (300, 80, 300, 1, False), (1165, 80, 512, 5, False), (300, 128, 300, 1, True),
    (300, 64, 300, 1, True), (700, 80, 700, 1, True), (182, 128, 43, 6, False), (2000, 128, 131, 6, True)])
def test_latent_heads_shared_by_prompts(tokens, heads, keys, prompts, shared):
    assert hip.mla_heads_shared(tokens, heads, keys, False, prompts) is shared


@pytest.mark.parametrize("m,n,k,reduced,takes", [
    # the next kernel sums the slabs (library / this, us): 8.5 / 5.5, 16.2 / 11.2; a small W at many rows 8.9 / 9.9, 10.2 / 13.3,
    # 17.7 / 16.5; 32 / 18; a router
    (1, 2048, 2048, False, True), (1, 6144, 4096, False, True), (128, 2048, 2048, False, False), (256, 2048, 2048, False, False),
    (256, 3072, 3072, False, False), (256, 4608, 3072, False, True), (16, 160, 6144, False, False),
    # with a reduction of its own: 26.7 / 28, 18.1 / 20; 41 / 33; 81 / 50; 11 / 21
    (1, 8192, 8192, True, False), (8, 6144, 6144, True, False), (48, 4096, 14336, True, True), (256, 8192, 8192, True, True),
    (256, 3072, 2048, True, False),
    # wide enough unsplit: 190 / 164, 309 / 252, 57 / 44
    (1, 128256, 4096, True, True), (256, 128256, 4096, True, True), (8, 32000, 4096, True, True),
    # above 256 rows: 316 / 186, 76 / 73, 94 / 97
    (512, 8192, 28672, True, True), (512, 8192, 8192, True, False), (512, 28672, 4096, True, False), (513, 8192, 28672, True, False)])
def test_short_batch_products(m, n, k, reduced, takes):
    assert hip.mid_profitable(m, n, k, reduced) is takes
    if takes:
        bm, bn, ksplit = hip.mid_choose(m, n, k, reduced)
        assert (bm, bn) in hip._MID_TILES and bm >= min(m, 256) and 1 <= ksplit <= k // 64


@pytest.mark.parametrize("m,n,k,reduced,takes,rows", [
    # library / this, us: 114 / 74, 107 / 90, 147 / 133, 45 / 31, 76 / 54, 219 / 161; tiles by the thousand, squarer shapes and more rows
    # (265 / 287, 165 / 143, 37 / 33, 97 / 101)
    (557, 4096, 14336, False, True, 192), (768, 4096, 14336, True, True, None), (1280, 4096, 14336, False, True, 256),
    (557, 2048, 8192, True, True, None), (300, 4096, 14336, False, True, 192), (300, 8192, 28672, False, True, 192),
    (640, 8192, 28672, False, False, None), (1281, 4096, 14336, False, False, None), (557, 4096, 4096, False, False, None),
    (557, 10240, 8192, True, False, None),
    # a small W of K = 2 N: 55 / 62 with a reduction of its own, 62 / 61 (and the norm) without; 62 / 50; 76 / 71
    (769, 3584, 7168, True, False, None), (769, 3584, 7168, False, True, None), (768, 3584, 7168, True, True, None),
    (769, 4096, 8192, True, True, None)])
def test_products_of_several_row_tiles(m, n, k, reduced, takes, rows):
    assert hip.mid_profitable(m, n, k, reduced) is takes
    if takes:
        bm, bn, ksplit = hip.mid_choose(m, n, k, reduced)
        assert bm >= 128 and ksplit > 1 and bm == (rows or bm)


@pytest.mark.parametrize("m,n,k,slow", [
    # us: 158 in tiles of 192 x 128 and 106 in 192 x 256, 154 and 100; in 16 splits and in 12 25.7 and 23.2, 21.0 and 18.7
    (257, 8192, 16384, (192, 128, 2)), (272, 8192, 16384, (192, 128, 2)), (160, 2048, 12288, (192, 128, 16)),
    (130, 2048, 8192, (192, 128, 16))])
def test_tiles_that_are_not_chosen(m, n, k, slow):
    assert hip.mid_profitable(m, n, k, False) and hip.mid_choose(m, n, k, False) != slow


def test_gate_up_at_short_batches():
    assert hip.mid_silu_profitable(1, 28672, 4096) and hip.mid_silu_profitable(256, 57344, 8192)
    assert not hip.mid_silu_profitable(257, 57344, 8192) and not hip.mid_silu_profitable(9, 28672, 2048)
    assert not hip.mid_silu_profitable(1, 7168, 8192)
    # 8 rows and a reduction below 4096: the barrier-free stream
    assert hip.stream_profitable(8, 28672, 2048) and not hip.stream_profitable(8, 28672, 4096)


def test_short_batch_products_are_planned_once_a_shape(monkeypatch):
    """A step outside a graph asks for the plan of every product several times over: only a shape's first answer is worked out."""
    asked = []
    real = hip._mid_estimate
    monkeypatch.setattr(hip, "_mid_estimate", lambda *a: (asked.append(a), real(*a))[1])

    def layer(m):                            # rows that no other test asks for
        plans = []
        for n, k in ((10224, 8128), (8176, 8128), (8176, 28608)):
            for reduced in (False, True):
                plans.append((hip.mid_profitable(m, n, k, reduced), hip.mid_choose(m, n, k, reduced)))
        return plans
    for m in (1, 101, 129, 250, 401):
        first = layer(m)
        assert asked, "the rule no longer asks the model of a product's time"
        asked.clear()
        assert layer(m) == first and not asked
    for rule in (hip.mid_choose, hip.mid_profitable, hip.mid_silu_tile):
        assert rule.cache_info().maxsize is not None          # (bounded)


def test_the_k_splits_to_choose_from_can_be_restricted():
    """VDAMD_MID_KSPLITS is read when the module is loaded; a switch that lost its meaning says so."""
    import os
    import subprocess
    import sys
    code = ("from vllm_distributed_amd.ops import hip\n"
            "print(sorted({hip.mid_choose(m, n, k)[2] for m in (1, 64, 256) for n, k in ((8192, 8192), (10240, 8192), (8192, 28672))}))")
    env = dict(os.environ, VDAMD_MID_KSPLITS="1,5", VDAMD_MID_GEMM_VARIANT="0",
               PYTHONPATH=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    got = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, check=True)
    assert got.stdout.strip().splitlines()[-1] in ("[5]", "[1, 5]")
    assert "VDAMD_MID_GEMM_VARIANT has no effect" in got.stdout + got.stderr


@pytest.mark.parametrize("batch,heads,kv_heads,dim,keys,once", [
    (48, 32, 8, 128, 13500, True), (48, 128, 8, 128, 13500, True), (3, 32, 8, 128, 13500, False), (48, 32, 8, 256, 13500, False),
    # the same keys in several workgroups, one for every 16 query heads of a key head (cached / past the caches: 141 / 174, 153 / 236)
    (48, 64, 2, 128, 13500, False), (200, 64, 2, 128, 4500, False), (100, 71, 1, 64, 13500, False), (48, 34, 2, 128, 13500, False)])
def test_decode_attention_reads_past_the_caches_what_one_workgroup_reads(batch, heads, kv_heads, dim, keys, once):
    assert hip.decode_reads_once(batch, heads, kv_heads, dim, keys) is once


@pytest.mark.parametrize("window,once", [(0, True), (257, True), (256, True), (255, False), (32, False)])
def test_decode_attention_past_the_caches_counts_the_keys_of_the_window(window, once, monkeypatch):
    import torch
    from vllm_distributed_amd import ops
    handed = []

    class Lib:
        @staticmethod
        def vdamd_paged_attention_decode(*args):
            handed.append(args[-2])
            return 0
    monkeypatch.setattr(hip, "_LIB", Lib)
    monkeypatch.setattr(hip, "_stream", lambda: None)
    monkeypatch.setattr(hip, "DECODE_ONCE_BYTES", 2 * 256 * 64 * 4)
    kc, vc = (torch.zeros(shape, dtype=torch.bfloat16) for shape in (ops.k_cache_shape(8, 1, 64, 64), ops.v_cache_shape(8, 1, 64, 64)))
    hip.paged_attention_decode(torch.zeros(2, 4, 64, dtype=torch.bfloat16), kc, vc, torch.zeros(2, 8, dtype=torch.int32),
                               torch.tensor([512, 3], dtype=torch.int32), 0.1, 512, num_splits=1, window=window)
    assert [past > 0 for past in handed] == [once]


def test_recurrent_layers_report_their_prompt_memory():
    """What a prompt through a recurrent layer allocates counts in the memory profile, which does not run its kernels."""
    import torch

    from vllm_distributed_amd import ops
    from vllm_distributed_amd.models.layers import linear_attention as la
    from vllm_distributed_amd.worker.model_runner import ModelRunner
    if not ops.hip_available():
        pytest.skip("the kernel library is not built")
    layers = [la.DecayLinearAttention(8, 64, 64, [0.9] * 8, 0), la.GatedDeltaRule(16, 8, 128, 128, 1),
              la.SelectiveStateSpace(8, 2, 64, 64, 2),
              la.GatedLinearHeads(256, 4, 64, 64, 16, 16.0, 1e-6, 3, torch.bfloat16)]
    # (rows + 63 for each sequence) / 64 chunks of 128 KB and more per head, and the fp32 result
    for layer, heads, vdim in zip(layers, (8, 16, 8, 4), (64, 128, 64, 64)):
        assert layer.prompt_bytes(16, 16) == 4 * 16 * heads * vdim                       # never chunked
        assert layer.prompt_bytes(2048, 32) > layer.prompt_bytes(2048, 1) > 32 * heads * 48 * 1024
        assert layer.prompt_bytes(1 << 17, 64) <= hip.CHUNK_SCRATCH_BYTES + 4 * (1 << 17) * heads * vdim
    runner = ModelRunner.__new__(ModelRunner)
    runner.model, runner.max_num_reqs, runner.is_gpu = torch.nn.ModuleList(layers + [torch.nn.Linear(2, 2)]), 32, True
    assert runner._prompt_bytes(2048) == layers[1].prompt_bytes(2048, 32) == max(m.prompt_bytes(2048, 32) for m in layers)
    runner.is_gpu = False
    assert runner._prompt_bytes(2048) == 0
