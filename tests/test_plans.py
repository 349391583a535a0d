"""The launch plans are plain functions of shapes: what the kernels' host checks rely on holds
for every shape (no empty split, whole chunks and pages, bounds on the number of splits)."""
import itertools
import os
import re
import subprocess

import pytest

from minfer_amd.kernels import ops


def test_skinny_plan_covers_k_without_empty_splits():
    for m, n, k, target in itertools.product((1, 8, 9, 16, 17, 40, 64), (96, 3584, 4608, 37888, 152064),
                                             (64, 200, 256, 3584, 8192, 18944), (64, 256, 1024)):
        splits, per = ops.skinny_plan(m, n, k, target_blocks=target)
        assert splits >= 1 and per % 256 == 0
        assert splits * per >= k, (m, n, k, splits, per)
        assert (splits - 1) * per < k, (m, n, k, splits, per)        # the last split has work
        if m <= 16 and k < 8192:
            assert splits == 1
        else:
            assert splits * ((n + 127) // 128) <= max(target, (n + 127) // 128), (m, n, k, splits)


def test_skinny_plan_choices_at_the_model_shapes():
    """At most 8 rows against a long K: one kernel where a CU's share of the weight rows fills its
    tiles (3584 and 8192 rows over 256 CUs), the staged K-split kernel where it does not (5120)."""
    assert ops.skinny_plan(8, 3584, 18944, target_blocks=256)[0] == 1
    assert ops.skinny_plan(8, 8192, 29568, target_blocks=256)[0] == 1
    assert ops.skinny_plan(1, 5120, 27648, target_blocks=256)[0] > 1
    assert ops.skinny_plan(9, 3584, 18944, target_blocks=256)[0] > 1
    assert ops.skinny_plan(16, 37888, 3584, target_blocks=256)[0] == 1
    # K of 8192 is held in registers where SwiGLU (or a norm) is folded in: one kernel up to 16 rows
    assert ops.skinny_plan(16, 59136, 8192, target_blocks=256, swiglu=True)[0] == 1
    assert ops.skinny_plan(16, 8192, 8192, target_blocks=256)[0] > 1
    assert ops.skinny_plan(12, 300, 8192, target_blocks=256, swiglu=True)[0] > 1      # too few weight rows for it


def test_tile_plan():
    """The tile product's plan for every shape is one the kernels take: a K split only for the
    variants that have one, in whole chunks of 256 with no empty part, the direct-to-LDS kernel only
    for K in 64s, no SwiGLU epilogue on the 192-wide tile."""
    for m, n, k, epi, aligned in itertools.product((65, 128, 200, 512, 1024, 2048, 5977, 8192), (96, 3584, 4608, 37888),
                                                   (64, 200, 256, 3584, 18944), (ops.EPI_F32, ops.EPI_SWIGLU),
                                                   (True, False)):
        if epi == ops.EPI_SWIGLU and n % 64:
            continue
        variant, splits, per = ops.tile_plan(m, n, k, epi, aligned and k % 8 == 0, n_cu=256)
        assert variant in (2, 9, 12, 13, 15)
        if variant in (12, 13, 15):
            assert aligned and k % 64 == 0
        assert variant != 15 or epi != ops.EPI_SWIGLU
        if splits == 1:
            assert per == k
            continue
        assert variant in (2, 12) and per % 256 == 0 and per >= 512
        assert splits * per >= k and (splits - 1) * per < k
        if variant == 12:
            assert m >= 768 and per >= 2048 and splits <= 8 and epi != ops.EPI_SWIGLU
        else:
            tiles = ((m + 127) // 128) * ((n + 127) // 128)
            assert tiles < 256 and splits * tiles <= 512


def test_split_plan_of_the_32_bit_attention():
    for n_tok, nk, group, hd, max_len in itertools.product((1, 8, 64, 300), (1, 2, 4), (1, 5, 7), (16, 128, 256),
                                                           (1, 64, 100, 4096, 32768)):
        n_splits, split_len = ops.split_plan(n_tok, nk, group, hd, max_len)
        assert 1 <= n_splits <= 64
        assert split_len % ops.PAGE == 0 and split_len > 0
        assert n_splits * split_len >= max_len
        assert (n_splits - 1) * split_len < max_len                   # the last split has keys


def test_decode_split_plan_bounds():
    for n_tok, nk, group, max_len in itertools.product((1, 8, 64, 300), (1, 2, 4), (1, 5, 7, 17), (1, 64, 4096, 32768)):
        places, n = ops.decode_split_plan(n_tok, nk, group, max_len, target_blocks=256)
        assert 1 <= n <= places <= 32
        assert n == 1 or n * 256 <= max_len + 255
        assert places == n or (1 < n_tok <= 64 and n > 1 and max_len >= 8192 and places == min(4 * n, 32))
    plan = lambda *a: ops.decode_split_plan(*a, target_blocks=256)
    assert plan(1, 4, 7, 32768) == (32, 32) and plan(64, 4, 7, 32768) == (1, 1)
    assert plan(8, 4, 7, 32768) == (32, 8)          # shares in proportion to the keys
    assert plan(8, 4, 7, 4096) == (8, 8)
    assert ops.decode_split_plan(8, 4, 7, 4096, target_blocks=64) == (2, 2)        # a chip of 64 CUs splits less


def test_where_64_x_64_tiles_take_a_short_k():
    """17 to 64 rows: one tile kernel over the whole of a short K, but not where a tile's chain outlasts the K-split kernels
    (few rows against few weight rows of 2,048; few rows against more than a tile a CU without SwiGLU)."""
    tiles = lambda m, n, k, **kw: ops.plan_linear(m, n, k, n_cu=256, **kw)["kernel"] == "tile_step_kernel<64,64>"
    for m, n, k in ((17, 512, 2048), (17, 2048, 2048), (24, 1024, 2048), (32, 2560, 2048), (48, 512, 2048), (17, 512, 1536)):
        assert not tiles(m, n, k, swiglu=True, tiled=True) and tiles(m, n, k, swiglu=True), (m, n, k)
    for m, n, k in ((64, 2048, 2048), (33, 4096, 2048), (17, 12288, 2048), (64, 512, 1536), (17, 2048, 1536), (17, 512, 896),
                    (40, 22016, 2048), (32, 17920, 1536), (17, 9728, 896)):
        assert tiles(m, n, k, swiglu=True, tiled=True) and tiles(m, n, k, swiglu=True), (m, n, k)
    for m, n, k in ((17, 24576, 768), (24, 20480, 1024), (32, 24576, 768)):
        assert not tiles(m, n, k, accumulate=True, tiled=True) and tiles(m, n, k, accumulate=True), (m, n, k)
    for m, n, k in ((48, 24576, 768), (64, 20480, 1024), (17, 24576, 256), (17, 16384, 768), (17, 512, 1024), (32, 1152, 896),
                    (24, 16448, 896), (32, 24576, 640)):
        assert tiles(m, n, k, accumulate=True, tiled=True) and tiles(m, n, k, accumulate=True), (m, n, k)


def test_tile_plan_of_k_not_in_64s():
    """A product that cannot be copied straight into LDS is cut over K where its own kernels gain by it: not for the cheap
    epilogues of a K of a thousand (200 x 8000 SwiGLU 21.2 us whole, 34.7 in two parts), for sums added to 32 bits at the
    same sizes, and for any epilogue against a long K."""
    splits = lambda m, n, k, epi: ops.tile_plan(m, n, k, epi, k % 8 == 0, n_cu=256)[1]
    for m, n, k in ((200, 8000, 1000), (128, 8000, 1000), (2048, 512, 1000), (300, 4096, 1000), (700, 512, 808), (65, 4096, 808),
                    (700, 4096, 2000)):
        assert splits(m, n, k, ops.EPI_SWIGLU) == 1, (m, n, k)
    for m, n, k in ((512, 3000, 1000), (1500, 1000, 1000), (700, 2000, 1000), (128, 12000, 1000), (300, 4096, 1000)):
        assert splits(m, n, k, ops.EPI_BF16) == 1, (m, n, k)
    for m, n, k in ((200, 200, 808), (128, 1000, 808), (65, 20000, 1000)):
        assert splits(m, n, k, ops.EPI_ACC_F32) > 1, (m, n, k)
    for epi in (ops.EPI_ACC_F32, ops.EPI_F32, ops.EPI_BF16, ops.EPI_SWIGLU):
        assert splits(128, 1024, 5000, epi) > 1 and splits(65, 4096, 18000, epi) > 1


def test_plan_linear_names_the_kernels_of_the_model_shapes():
    """Which kernel a product takes, as the library decides it (nothing is launched): the decode
    shapes of the 7B, 32B and 72B widths get the kernels the design describes, and widths off the
    family's (896, 1024, 2560, 6144) a named path of their own."""
    p = lambda *a, **k: ops.plan_linear(*a, n_cu=256, **k)["kernel"]
    for h, inter, qkv in ((3584, 18944, 4608), (5120, 27648, 7168), (8192, 29568, 10240)):
        for m in (1, 8, 16):
            assert p(m, qkv, h, normed=True) == "stationary16_kernel(norm)"
            assert p(m, 2 * inter, h, swiglu=True, normed=True) == "stationary16_kernel(norm)"
            assert p(m, 152064, h, normed=True) == "stationary16_kernel(norm)"
        assert p(8, h, h, accumulate=True) == ("stationary16_kernel" if h <= 5120 else "rolling16_kernel")
        assert p(64, 2 * inter, h, swiglu=True) == "panel_kernel" and p(64, 152064, h) == "panel_kernel"
        # the ring form needs K in whole chunks of 256 (29568 is 115.5 of them)
        assert p(64, h, inter, accumulate=True) == ("skinny_ring_kernel" if inter % 256 == 0 else "skinny_kernel")
        assert p(2048, 2 * inter, h, swiglu=True) == "tile_dma_kernel<256>"
        assert p(40, qkv, h, normed=True) == ""                       # no fold above 16 rows: norm, then product
    assert p(8, 3584, 18944, accumulate=True) == "rolling16_kernel"
    # a prompt of 2,048 tokens at the 7B widths: 256-wide tiles of q|k|v (144) and o (112) would leave
    # half of the 256 CUs idle, so 192 tiles of 256 x 192 and 224 of 256 x 128; down has K to split
    assert p(2048, 4608, 3584, out_bf16=True) == "tile_dma_kernel<192>"
    assert p(2048, 3584, 3584, accumulate=True) == "tile_dma_kernel<128>"
    assert p(2048, 3584, 18944, accumulate=True) == "tile_dma_kernel<256>(split K)"
    assert p(8192, 4608, 3584, out_bf16=True) == "tile_dma_kernel<192>"       # 768 tiles: three whole rounds
    assert p(4096, 3584, 3584, accumulate=True) == "tile_dma_kernel<256>"     # 224 tiles: one round nearly full
    assert p(4096, 37888, 3584, swiglu=True) == "tile_dma_kernel<256>"
    assert p(2048, 3584, 3584 + 8, accumulate=True) == "tile_kernel<128,128>"      # K not in 64s
    assert p(200, 3584, 18944, accumulate=True) == "tile_dma_kernel<128>(split K)"
    # other widths: multiples of 256 that are instantiated take the register-resident kernel, the
    # rest the rolling one; unaligned operands the guarded ones
    for k in (1024, 2560, 3072, 6144, 7168):
        assert p(4, 4096, k, normed=True) == "stationary16_kernel(norm)", k
    # a width of 896 (the narrowest model of the family) runs as seven waves of four steps
    assert p(4, 4096, 896, normed=True) == "stationary16_kernel(norm)" and p(4, 4096, 896) == "stationary16_kernel"
    assert p(4, 4096, 640, normed=True) == "" and p(4, 4096, 640) == "rolling16_kernel"
    assert p(4, 4096, 1280) == "rolling16_kernel"                       # 5 x 256: not instantiated
    assert p(4, 4096, 900, aligned=False) == "skinny16_kernel"
    assert p(4, 100, 1024) == "rolling16_kernel"                        # too few weight rows to go round
    assert p(30, 4096, 900, aligned=False) == "skinny_kernel"
    for ns in ops.STATIONARY_NS:
        assert ops.stationary_shape(4096, 256 * ns, True) and p(2, 4096, 256 * ns, normed=True) != ""
    assert not ops.stationary_shape(4096, 256 * 5) and not ops.stationary_shape(4096, 256 * 33, True)


def test_shared_query_tiles_cover_every_page_once():
    """The host's list of workgroups for the prompt attention: every block of 128 queries appears
    with all its shares or alone, a share's pages are at most the load asked for (unless the cap on
    shares binds), the longest entries come first, and without long blocks there is no list."""
    import torch
    from minfer_amd.engine.batch import StepContext

    def ctx(new, start):
        n = sum(new)
        return StepContext(cache=None, n_tokens=n, n_seqs=len(new), token_ids=torch.zeros(n, dtype=torch.int32),
                           positions=None, seq_of_tok=None, cu_seqlens=None, start_pos=None, slot_ids=None,
                           logit_rows=None, page_tables={}, max_len=0, max_new=max(new), all_decode=False,
                           host_new=list(new), host_start=list(start))

    for new, start, window, load, cap in (([1500, 260, 40], [600, 0, 0], 0, 4, 8), ([64], [30000], 0, 26, 8),
                                          ([2048], [0], 0, 15, 8), ([300, 17], [900, 5000], 700, 4, 3)):
        got = ctx(new, start).shared_query_tiles(128, 64, window, 1, 1 << 19, 2, load, cap)      # the least load binds
        assert got is not None
        seqs, q0s, words, n_slots, most = (x.tolist() if hasattr(x, "tolist") else x for x in got)
        tiles = {}
        for b, q0, w in zip(seqs, q0s, words):
            tiles.setdefault((b, q0), []).append(w)
        assert sorted(tiles) == sorted((b, q0) for b, n in enumerate(new) for q0 in range(0, n, 128))
        slots = set()
        for (b, q0), ws in tiles.items():
            last_key = start[b] + min(q0 + 128, new[b]) - 1
            first_key = max(0, start[b] + q0 - window + 1) if window else 0
            pages = last_key // 64 - first_key // 64 + 1
            if ws == [0]:
                assert pages <= load
                continue
            n = (ws[0] >> 8) & 255
            assert sorted(w & 255 for w in ws) == list(range(n)) and {(w >> 8) & 255 for w in ws} == {n}
            assert len({w >> 16 for w in ws}) == 1 and 2 <= n <= min(cap, most)
            assert n == cap or -(-pages // n) <= load
            slots.add(ws[0] >> 16)
        assert slots == set(range(n_slots))
    assert ctx([100, 30], [0, 0]).shared_query_tiles(128, 64, 0, 1, 1 << 19, 2, 4, 8) is None
    # the even share binds: 64 tokens on 30,000 are 470 pages; 28 heads over 512 workgroups at once
    # give each at most 26 of them, 4 heads give each at most 4: layers with other head counts get
    # plans of their own from the same step
    c = ctx([64], [30000])
    a = c.shared_query_tiles(128, 64, 0, 28, 256, 2, 4, 64)
    b = c.shared_query_tiles(128, 64, 0, 4, 256, 2, 4, 64)
    assert a[4] == -(-470 // 26) and b[4] == 64 and c.shared_query_tiles(128, 64, 0, 28, 256, 2, 4, 64) is a
    # no sharing where it cannot gain: a whole prompt of 2,048 tokens with 28 heads keeps every CU
    # busy for as long as its longest block takes (32 pages against an even 30 a CU); with 2 heads
    # the CUs would idle behind the longest blocks
    assert ctx([2048], [0]).shared_query_tiles(128, 64, 0, 28, 256, 2, 4, 8) is None
    assert ctx([2048], [0]).shared_query_tiles(128, 64, 0, 2, 256, 2, 4, 8) is not None
    assert ctx([128] * 8, [2000] * 8).shared_query_tiles(128, 64, 0, 28, 256, 2, 4, 8) is None
    assert ctx([512], [4096]).shared_query_tiles(128, 64, 0, 28, 256, 2, 4, 8) is not None


def test_prefill_tile_takes_a_group_of_heads_together():
    """Rows of the prompt attention are (token, head of the kv group) pairs, 128 a workgroup: as many
    whole tokens as fit beside all heads of the group; a group with more heads than rows goes in chunks."""
    assert ops.prefill_tile(28, 4, 128) == (18, 7, 4)          # the 7B shape: 126 of 128 rows in use
    assert ops.prefill_tile(6, 6, 64) == (128, 1, 6)           # one head a group: 128 tokens
    assert ops.prefill_tile(64, 8, 128) == (16, 8, 8)
    assert ops.prefill_tile(40, 8, 256) == (25, 5, 8)
    assert ops.prefill_tile(130, 1, 16) == (1, 128, 2)         # 130 heads: a token's heads in two workgroups
    for nh, nk, hd in itertools.product((1, 3, 12, 28, 64, 300), (1, 2, 4), (16, 48, 128, 256)):
        if nh % nk:
            continue
        tq, gh, per_tile = ops.prefill_tile(nh, nk, hd)
        group = nh // nk
        assert 1 <= gh <= group and tq >= 1 and tq * gh <= 128
        assert per_tile == nk * -(-group // gh)


def test_skinny_plan_keeps_a_small_matrix_in_one_kernel():
    assert ops.skinny_plan(8, 2048, 11008, target_blocks=256, tiled=True)[0] == 1      # the 3B shape's down product
    assert ops.skinny_plan(16, 2048, 11008, target_blocks=256, tiled=True)[0] > 1
    assert ops.skinny_plan(8, 5120, 13824, target_blocks=256, tiled=True)[0] > 1       # the 14B shape's: 141 MB


def test_capped_form_of_wide_heads():
    """Heads too wide for two waves a SIMD (192 and more of keys and values together in pairs): no form of four waves where
    there are walks for every SIMD anyway, one head a wave where two would not fit a SIMD at all; narrow heads keep four waves."""
    form = lambda tiles, h, kv, d, v, mean, most: ops.capped_form(tiles, h, kv, d, v, mean, most, n_cu=256)
    for d, v in ((192, 192), (256, 128), (128, 256), (160, 160)):
        assert form(16 * 63, 16, 2, d, v, 500, 1000) == (2, 1)          # sixteen prompts of 1,000 tokens
        assert form(128, 16, 2, d, v, 512, 512) == (2, 1)               # 2,048 tokens, a window of 512: one round
        assert form(63, 16, 2, d, v, 500, 1000) == (2, 4)               # 1,000 tokens
        assert form(13, 16, 16, d, v, 102, 203)[0] == 1
    assert form(63, 16, 2, 256, 256, 500, 1000)[0] == 1 and form(63, 16, 2, 224, 224, 500, 1000)[0] == 2
    assert form(63, 16, 2, 128, 128, 500, 1000) == (2, 4) and form(63, 16, 16, 128, 128, 500, 1000) == (1, 4)
    assert form(16 * 63, 32, 4, 256, 64, 500, 1000) == (4, 1) and form(16 * 63, 32, 4, 256, 128, 500, 1000) == (2, 1)


def test_capped_form_of_short_and_even_walks():
    """Where there are walks for every SIMD and few keys to each, four waves a tile pay for their starts and ends: one or two;
    long walks and launches that leave SIMDs idle keep four, and four heads a wave are for keys twice as wide as values."""
    form = lambda tiles, h, kv, d, v, mean, most: ops.capped_form(tiles, h, kv, d, v, mean, most, n_cu=256)
    assert form(32 * 13, 16, 2, 64, 64, 100, 200)[1] < 4 and form(32 * 13, 16, 16, 128, 128, 100, 200)[1] < 4
    assert form(256, 16, 2, 64, 64, 200, 200) == (2, 1) and form(512, 12, 4, 128, 128, 100, 100)[1] < 4      # decode, no splits
    assert form(16 * 63, 16, 2, 128, 128, 500, 1000) == (2, 2) and form(16 * 63, 16, 16, 128, 128, 500, 1000) == (1, 1)
    assert form(16 * 63, 32, 4, 128, 128, 500, 1000) == (2, 2)
    for tiles, mean, most in ((13, 102, 203), (63, 500, 1000), (128, 1024, 2048), (24, 800, 1010)):
        assert form(tiles, 16, 2, 128, 128, mean, most) == (2, 4) and form(tiles, 8, 8, 64, 64, mean, most) == (1, 4)


def test_keys_in_sight():
    """Mean and most keys of a step's new tokens, against a count over the tokens."""
    import torch
    from minfer_amd.engine.batch import StepContext
    for new, start, window in (([5, 300], [0, 40], 0), ([100], [0], 64), ([7, 900], [500, 30], 128), ([1, 1], [10, 99], 50)):
        n, top = sum(new), max(a + b for a, b in zip(new, start))
        c = StepContext(cache=None, n_tokens=n, n_seqs=len(new), token_ids=torch.zeros(n, dtype=torch.int32), positions=None,
                        seq_of_tok=None, cu_seqlens=None, start_pos=None, slot_ids=None, logit_rows=None, page_tables={},
                        max_len=top, max_new=max(new), all_decode=False, host_new=list(new), host_start=list(start))
        keys = [min(s + i + 1, window or top) for k, s in zip(new, start) for i in range(k)]
        mean, most = c.keys_in_sight(window)
        assert abs(mean - sum(keys) / n) < 0.5 and most == min(top, window or top)
        assert c.keys_in_sight(0, 64)[0] <= 32 and c.keys_in_sight(0, 64)[1] == min(top, 64)


# the sizes at which two heads a wave stop to fit 256 registers, and 512; one head at the largest
@pytest.mark.parametrize("dim,v_dim", [(128, 128), (192, 80), (160, 160), (192, 192), (256, 128), (224, 224), (256, 256)])
def test_capped_forms_keep_to_their_registers(dim, v_dim):
    """The compiler's own report of the matrix-core attention: of the forms that a plan may choose at a size (heads a wave up
    to what `capped_form` takes, any number of waves), none with one or two heads spills a register."""
    from minfer_amd.kernels import build
    flags = [f for f in build.HIPCC_FLAGS if f != "-shared"]
    out = subprocess.run([build._hipcc(), *flags, f"-DMF_CAPM_D={dim}", f"-DMF_CAPM_V={v_dim}", "-I", build.CSRC, "-c", "--cuda-device-only",
                          "-Rpass-analysis=kernel-resource-usage", os.path.join(build.CSRC, "attn_capped_mfma.hip"), "-o", os.devnull],
                         capture_output=True, text=True)
    assert out.returncode == 0, out.stderr[-2000:]
    spills, form = {}, None
    for line in out.stderr.splitlines():
        if "Function Name" in line:
            m = re.search(r"capped_mfma_kernelILi(\d)ELi(\d)E", line)
            form = (int(m.group(1)), int(m.group(2))) if m else None
        elif form and "VGPRs Spill:" in line:
            spills[form] = int(re.search(r"VGPRs Spill: (\d+)", line).group(1))
    heads = ops.capped_form(13, 2, 1, dim, v_dim, 100, 203, n_cu=256)[0]
    assert (heads, 1) in spills and (heads, 4) in spills and (1, 4) in spills
    assert not {f: n for f, n in spills.items() if f[0] <= heads and n}, spills


def test_tile_plan_has_one_price_for_whole_and_cut():
    """Few tiles against a K around the end of the 64 x 64 tiles' own price: a product that is cut at either end of a run of neighbouring
    K is cut in between as well (whole, 88 x 896 would be 28 workgroups on 256 CUs, each with the whole chain over K)."""
    for m, n, epi in itertools.product((65, 88, 100, 128), (256, 512, 896, 1024, 1536, 2048, 2560, 3200),
                                       (ops.EPI_F32, ops.EPI_ACC_F32, ops.EPI_BF16, ops.EPI_SWIGLU)):
        ks = range(2944, 3648, 64)
        cut = [ops.tile_plan(m, n, k, epi, True, n_cu=256)[1] > 1 for k in ks]
        first, last = cut.index(True), len(cut) - cut[::-1].index(True)
        assert all(cut[first:last]), (m, n, epi, [k for k, c in zip(ks, cut) if not c])
    for m, n in ((88, 896), (100, 3200), (128, 2560)):
        for k in range(3072, 3329, 64):
            assert ops.tile_plan(m, n, k, ops.EPI_ACC_F32, True, n_cu=256)[1] > 1, (m, n, k)


def test_tile_plan_of_a_short_k():
    """The plans that `test_tile_plan` holds the long and the shortest K to, where the 64 x 64 tiles have their own price and a split is
    credited with what the kernel behind the product saves: whole chunks, no empty part, K in 64s."""
    for m, n, k, epi, behind in itertools.product((65, 100, 203, 445, 604, 1024, 2048), (96, 896, 1152, 2048, 4608, 8192),
                                                  (512, 896, 1536, 2048, 3008, 3072, 3136, 3200, 3264, 3328), (ops.EPI_F32, ops.EPI_ACC_F32),
                                                  (0, 1, 2)):
        variant, splits, per = ops._tile_plan(m, n, k, epi, True, 256, behind)
        assert variant in (2, 12, 13, 15, 16)
        if splits == 1:
            assert per == k
            continue
        assert variant in (2, 12) and per % 256 == 0 and per >= 512
        assert splits * per >= k and (splits - 1) * per < k
        tiles = ((m + 127) // 128) * ((n + 127) // 128)
        assert variant == 12 or (tiles < 256 and splits * tiles <= 512)


def test_where_an_activation_joins_its_product():
    """An expert that every token takes, 4,096 gates and ups of 2,048 and a logit's rows: the activation in the epilogue only from the rows
    on where the tiles that have it, and the logits' own product, cost less than the plain product's tiles and the activation's kernel."""
    pays = lambda m, f, k: ops.linear_gated_pays(m, f, 2 * f + 16, k, n_cu=256)
    for m in (65, 96, 128, 160, 203, 256, 300, 384):
        assert not pays(m, 4096, 2048), m
    for m in (512, 1024, 2048, 4096):
        assert pays(m, 4096, 2048), m
    for m, f, k in ((65, 1024, 2048), (768, 1024, 2048), (1024, 768, 1024), (1024, 512, 2048), (256, 2048, 1024), (65, 4096, 4096), (64, 4096, 2048),
                    (1, 4096, 2048)):
        assert not pays(m, f, k), (m, f, k)
    for m, f, k in ((2048, 1024, 2048), (2048, 4096, 4096), (1024, 2048, 1024)):
        assert pays(m, f, k), (m, f, k)
    assert pays(8192, 1024, 2048) and pays(20000, 5632, 2048)


def test_last_weight_rows_apart_whatever_the_epilogue():
    """A rest of a few weight rows is a launch of its own for every epilogue that takes its columns one by one."""
    for epi in (ops.EPI_F32, ops.EPI_ACC_F32, ops.EPI_BF16, ops.EPI_RELU2):
        for m, n, k in ((2048, 8224, 2048), (2048, 8200, 4096), (4096, 8208, 2048)):
            assert ops.tile_plan(m, n, k, epi, n_cu=256)[0] == 16, (m, n, k, epi)
    for epi in (ops.EPI_XIELU, ops.EPI_SWIGLU):
        assert ops.tile_plan(2048, 8256, 2048, epi, n_cu=256)[0] != 16


def test_plan_linear_names_the_kernels_of_folded_norms():
    """The kernel that a product takes with a norm folded in on either side, "" where `linear_fused` declines; and how a product of many
    rows is cut where the kernel behind it adds its parts."""
    p = lambda *a, **k: ops.plan_linear(*a, n_cu=256, **k)["kernel"]
    both = dict(scale_in=True, norm_out=True)
    for m, n, k in ((17, 1152, 896), (20, 896, 4864), (64, 2048, 2048), (33, 2048, 1536), (32, 3072, 3072)):
        for kw in (dict(scale_in=True), dict(norm_out=True), both):
            assert p(m, n, k, accumulate=True, **kw) == p(m, n, k, tiled=True, **kw) == "whole_kernel", (m, n, k, kw)
        assert p(m, n, k, accumulate=True) != "whole_kernel"
        assert p(m, n, k, scale_in=True, out_bf16=True) != "whole_kernel"
        assert p(m, n + 8, k, norm_out=True) != "whole_kernel"
    assert p(17, 1152 + 8, 896, scale_in=True) == p(40, 1001, 1024, scale_in=True) == "tile_step_kernel<64,64>"
    assert p(64, 3584, 3584, norm_out=True) == p(64, 3584, 18944, norm_out=True) == "skinny_ring_kernel"
    assert p(64, 37888, 3584, swiglu=True, scale_in=True) == "panel_kernel" and p(64, 40960, 3584, norm_out=True) == ""
    assert p(8, 3584, 18944, norm_out=True, tiled=True) == "rolling16_kernel" and p(8, 3584, 18944, scale_in=True, tiled=True) == ""
    assert p(8, 3584, 3584, **both) == "stationary16_kernel"
    for m, n, k in ((8, 300, 200), (20, 300, 200), (64, 64, 256)):
        assert p(m, n, k, norm_out=True) == "" and p(m, n, k, scale_in=True) == "", (m, n, k)
    for bad in (dict(norm_out=True, out_bf16=True), dict(norm_out=True, swiglu=True)):
        with pytest.raises(ops.KernelError):
            ops.plan_linear(32, 1024, 896, n_cu=256, **bad)
    for (m, n, k), behind in (((100, 1152, 896), 1), ((300, 896, 896), 2), ((200, 2048, 2048), 1)):
        assert ops.plan_linear(m, n, k, n_cu=256)["splits"] == 1
        cut = ops.plan_linear(m, n, k, n_cu=256, behind=behind)
        assert cut["splits"] > 1 and cut["kernel"].endswith("(split K)")


def test_tile_plan_with_the_tiled_copy():
    """With the tiled copy a product takes the plan that it takes without, or the kernel that reads that copy alone: never for SwiGLU, for up
    to 128 rows or a K not in 64s; all its tiles on the chip at once, at most eight parts, none of them empty."""
    taken = 0
    for n_cu, m, n, k, behind in itertools.product((104, 256), (65, 128, 129, 203, 300, 604, 900, 2048), (96, 512, 1001, 2048, 8192),
                                                   (64, 200, 2048, 3648, 18944), (0, 1, 2)):
        for epi in (ops.EPI_ACC_F32, ops.EPI_SWIGLU):
            if epi == ops.EPI_SWIGLU and n % 64:
                continue
            plain, (variant, splits, per) = (ops._tile_plan(m, n, k, epi, k % 8 == 0, n_cu, behind, t) for t in (False, True))
            if (variant, splits, per) == plain:
                assert variant <= 20
                continue
            taken += 1
            assert variant in (26, 28) and epi != ops.EPI_SWIGLU and m > 128 and k % 64 == 0
            bm = (variant - 20) * 16
            assert (m + bm - 1) // bm * ((n + 127) // 128) * splits <= n_cu and 1 <= splits <= 8
            assert per == k if splits == 1 else per % 64 == 0 and (splits - 1) * per < k <= splits * per
    assert taken > 50


def test_stream_plan_follows_tiles_and_results():
    """Which kernel a product takes with the tiled copy follows from prices: along the rows it changes where a tile is added (tiles have 64 to 256
    rows in 32s), and between two such numbers where one price passes another, which is another number for every shape.  (Lines at 700 and 1,100
    rows were the same two numbers for most of these.)"""
    changes = {}
    for n, k, behind in itertools.product((512, 768, 896, 1024), (2048, 3072, 4864, 8192), (0, 2)):
        plans = [ops._tile_plan(m, n, k, ops.EPI_ACC_F32 if behind else ops.EPI_F32, True, 256, behind, True)[0] > 20 for m in range(129, 1409)]
        for i in range(1, len(plans)):
            if plans[i] != plans[i - 1]:
                changes.setdefault(129 + i, []).append((n, k, behind))
    assert changes
    assert not {m: at for m, at in changes.items() if m % 32 != 1 and len(at) > 2}


@pytest.mark.parametrize("m,n,k", [(1400, 1536, 320), (1400, 1536, 512), (3169, 896, 4864), (3379, 896, 4864), (2721, 1024, 4096), (3995, 768, 3072), (3281, 640, 2560), (4310, 640, 2560), (3372, 1000, 2816)])
def test_stream_plan_in_front_of_the_norm(m, n, k):
    """A K of a few hundred; and thousands of rows against few weight rows: whole in `tile_stream_kernel` with a norm kernel behind it they took 2 to 12 % longer than in the
    parts that the kernel with the norm adds."""
    assert ops._tile_plan(m, n, k, ops.EPI_ACC_F32, True, 256, 2, True) == ops._tile_plan(m, n, k, ops.EPI_ACC_F32, True, 256, 2, False)
