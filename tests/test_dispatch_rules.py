"""Rules that choose between two forms of an operation, at sizes where both were timed (us on one MI355X, issued one
after the other from Python): the form chosen takes at most 1.15 times the other's time."""
import pytest

from fasttalk_llm_microservice_amd.ops import mixers as M


def segments(rows, count, pos):
    start = [i * rows for i in range(count + 1)]
    return M.Segments(None, None, None, None, None, count, rows, pos + rows, host=(start, [pos] * count, [pos + rows] * count))


CAUSAL = dict(heads=16, kv_heads=4, dk=128, dv=128, window=0)
SPECS = {
    "plain": CAUSAL, "cap": dict(CAUSAL, softcap=30.0), "table": dict(CAUSAL, dist_bias=True),
    "sigmoid": dict(CAUSAL, sigmoid=True), "narrow": dict(heads=8, kv_heads=8, dk=64, dv=64, window=0),
    "window": dict(CAUSAL, window=1024), "two maps": dict(CAUSAL, dk=64, window=1024, maps=2),
    "wide blocks": dict(heads=16, kv_heads=16, dk=128, dv=128, window=4096, blocks=True), "terms": dict(CAUSAL, r1=True),
    "sigmoid terms": dict(CAUSAL, sigmoid=True, r1=True), "cap table": dict(CAUSAL, softcap=30.0, dist_bias=True),
}


@pytest.mark.parametrize("spec,rows,count,pos,one,products", [
    ("plain", 32, 1, 0, 11, 118), ("plain", 32, 1, 2000, 54, 122), ("plain", 64, 1, 8000, 174, 144),
    ("plain", 64, 1, 30000, 609, 566), ("plain", 300, 1, 4000, 101, 245), ("plain", 300, 1, 30000, 623, 1937),
    ("plain", 1000, 1, 30000, 664, 5150), ("plain", 2000, 1, 0, 72, 510), ("plain", 40, 8, 700, 29, 806),
    ("plain", 32, 4, 15000, 312, 771), ("plain", 33, 1, 120000, 2381, 1599), ("cap", 64, 1, 8000, 258, 142),
    ("cap", 300, 1, 4000, 145, 243), ("cap", 32, 4, 15000, 463, 780), ("table", 32, 1, 2000, 65, 116),
    ("table", 64, 1, 30000, 771, 617), ("table", 1000, 1, 30000, 801, 5784), ("sigmoid", 32, 1, 2000, 66, 104),
    ("sigmoid", 64, 1, 30000, 806, 478), ("sigmoid", 32, 4, 15000, 408, 650), ("sigmoid", 1000, 1, 30000, 839, 3703),
    ("sigmoid", 300, 1, 0, 22, 108), ("narrow", 64, 1, 8000, 119, 128), ("narrow", 300, 1, 4000, 70, 169),
    ("narrow", 64, 1, 30000, 412, 338), ("narrow", 1000, 1, 30000, 429, 2111), ("window", 64, 1, 8000, 34, 105),
    ("window", 300, 1, 4000, 36, 139), ("two maps", 64, 1, 8000, 29, 108), ("wide blocks", 64, 1, 8000, 91, 103),
    ("wide blocks", 300, 1, 4000, 95, 259), ("wide blocks", 2000, 1, 0, 72, 441), ("plain", 64, 1, 4000, 93, 103),
    ("plain", 128, 1, 8000, 173, 227), ("plain", 128, 1, 30000, 607, 746), ("plain", 32, 1, 8000, 172, 124),
    ("plain", 100, 1, 3000, 75, 119), ("cap", 64, 1, 4000, 137, 106), ("cap", 128, 1, 8000, 259, 229),
    ("cap", 200, 1, 8000, 260, 384), ("cap", 32, 1, 2000, 74, 107), ("table", 64, 1, 8000, 219, 149),
    ("table", 128, 1, 8000, 219, 232), ("sigmoid", 64, 1, 8000, 223, 122), ("sigmoid", 128, 1, 8000, 227, 196),
    ("sigmoid", 250, 1, 20000, 549, 687), ("narrow", 64, 1, 4000, 66, 97), ("narrow", 128, 1, 8000, 121, 136),
    ("narrow", 200, 1, 8000, 121, 189), ("terms", 64, 1, 8000, 325, 135), ("terms", 300, 1, 4000, 181, 245),
    ("sigmoid terms", 64, 1, 8000, 270, 119), ("sigmoid terms", 300, 1, 4000, 152, 216),
    ("cap table", 64, 1, 8000, 564, 146), ("cap table", 300, 1, 4000, 311, 258), ("plain", 64, 4, 8000, 174, 520),
    ("cap", 2000, 1, 8000, 572, 2913), ("plain", 48, 16, 1500, 49, 1428)])
def test_long_windowed_segments(spec, rows, count, pos, one, products):
    sp = M.WindowSpec(scale=1.0, **SPECS[spec])
    taken = one if M._band_pays(segments(rows, count, pos), sp, 32) else products
    assert taken <= 1.15 * min(one, products)


@pytest.mark.parametrize("act,n,k,rows,few,vendor", [
    (None, 2048, 2048, 1, 5.4, 11.1), (None, 2048, 2048, 64, 8.8, 11.7), (None, 2048, 8192, 48, 21.8, 15.1),
    (None, 5120, 13824, 1, 47.7, 29.7), (None, 5120, 13824, 32, 56.8, 36.8), (None, 13824, 5120, 16, 42.9, 27.7),
    (None, 14336, 4096, 1, 24.0, 29.0), (None, 14336, 4096, 32, 37.6, 26.2), (None, 8192, 2048, 16, 10.3, 13.3),
    (None, 6144, 2048, 64, 18.6, 13.1), (None, 32768, 2048, 32, 27.7, 34.1), (None, 256, 2048, 64, 6.7, 5.3),
    (None, 512, 16384, 64, 45.4, 19.1), (None, 20480, 5120, 17, 58.7, 42.1), ("silu", 16384, 2048, 16, 14.9, 21.1),
    ("silu", 4096, 8192, 1, 31.7, 19.6), ("silu", 4096, 8192, 64, 37.7, 28.2), ("silu", 28672, 4096, 64, 68.3, 54.2),
    ("silu", 28672, 4096, 16, 49.4, 63.0), ("clamp_glu", 2048, 2048, 64, 13.0, 14.6),
    ("relu_sq", 8192, 2048, 64, 19.1, 16.2), ("relu_sq", 8192, 2048, 32, 11.8, 15.4),
    ("relu_sq", 14336, 4096, 32, 38.1, 27.7), ("relu_sq", 2048, 8192, 48, 21.7, 17.5),
    ("relu_sq", 2048, 8192, 1, 11.7, 15.1)])
def test_products_of_few_rows(act, n, k, rows, few, vendor):
    taken = few if M._few_rows_pays(rows, n, k, act) else vendor
    # (the kernel's times alone; its call is 15 us cheaper on the host)
    assert taken <= max(1.15 * min(few, vendor), vendor + 1.5)


@pytest.mark.parametrize("experts,top,ff,width,shared,rows,few,pairs", [
    (32, 4, 1536, 2048, False, 1, 32.0, 24.9), (32, 4, 1536, 2048, False, 4, 56.8, 46.2), (32, 4, 1536, 2048, False, 8, 70.8, 70.6),
    (32, 4, 1536, 2048, False, 32, 92.8, 214.0), (32, 4, 1536, 2048, True, 1, 43.7, 41.7), (32, 6, 1024, 2048, True, 2, 62.0, 67.5),
    (128, 8, 768, 2048, False, 4, 86.5, 74.4), (128, 8, 768, 2048, False, 16, 163.4, 204.5), (8, 2, 4096, 4096, False, 1, 50.0, 40.2),
    (8, 2, 4096, 4096, False, 6, 136.7, 183.8), (8, 2, 14336, 4096, False, 1, 158.0, 138.2), (8, 2, 14336, 4096, False, 4, 436.5, 462.7),
    (256, 8, 256, 1024, False, 8, 52.4, 46.5), (256, 8, 256, 1024, False, 48, 112.7, 137.3), (16, 2, 2048, 6144, False, 4, 126.5, 111.6),
    (16, 2, 2048, 6144, False, 16, 214.4, 356.3), (64, 8, 1408, 4096, False, 1, 110.2, 83.9), (64, 8, 1408, 4096, False, 8, 271.9, 344.8),
    (4, 1, 512, 512, False, 8, 14.1, 11.4), (4, 1, 512, 512, False, 64, 15.6, 22.5)])
def test_experts_of_few_rows(experts, top, ff, width, shared, rows, few, pairs):
    taken = few if M.experts_few_pays(rows * top, experts, ff * width, shared) else pairs
    assert taken <= 1.15 * min(few, pairs)


@pytest.mark.parametrize("experts,one,two", [(16, 6.3, 14.7), (32, 10.3, 16.7), (64, 15.4, 17.5), (128, 25.2, 20.4)])
def test_grouped_softmax_router(experts, one, two):
    assert (one if M.moe_route_softmax_pays(experts) else two) == min(one, two)


def unlike(lens):
    start = [0]
    for n in lens:
        start.append(start[-1] + n)
    return M.Segments(None, None, None, None, None, len(lens), max(lens), host=(start, [5] * len(lens), [n + 5 for n in lens]))


@pytest.mark.parametrize("heads,dk,dv,lens,chunks,walks", [
    (16, 128, 128, [100] * 64, 554, 1057), (16, 128, 128, [96], 51, 61), (32, 64, 64, [100] * 16, 124, 113),
    (32, 64, 64, [100] * 64, 489, 403), (32, 64, 64, [256] * 32, 472, 497), (32, 64, 64, [2000] * 4, 471, 793),
    (4, 128, 256, [100] * 64, 212, 487), (32, 16, 32, [100] * 64, 264, 130), (32, 16, 32, [256] * 32, 266, 168),
    (32, 16, 32, [777], 55, 181), (32, 16, 32, [2000] * 4, 277, 542), (32, 64, 64, [1] * 64 + [4000], 475, 1455)])
def test_delta_rule_of_long_segments(heads, dk, dv, lens, chunks, walks):
    taken = chunks if M._delta_chunks_pay(unlike(lens), heads, dk, dv) else walks
    assert taken <= 1.1 * min(chunks, walks)


@pytest.mark.parametrize("heads,n,dv,lens,chunks,walks", [
    (16, 128, 128, [256] * 32, 420, 388), (16, 128, 128, [777], 59, 170), (16, 128, 128, [2000] * 4, 371, 459),
    (16, 128, 128, [256] * 4, 64, 67), (32, 64, 64, [300] * 8, 82, 74), (32, 64, 64, [256] * 32, 193, 201),
    (4, 128, 256, [300] * 8, 95, 78), (4, 128, 256, [2000] * 4, 183, 425), (32, 16, 32, [256] * 32, 99, 87),
    (32, 16, 32, [300] * 8, 44, 49), (16, 128, 128, [1] * 32 + [400], 103, 125), (32, 16, 32, [4096], 77, 564)])
def test_state_space_scan_of_long_segments(heads, n, dv, lens, chunks, walks):
    taken = chunks if M._ssd_chunks_pay(unlike(lens), heads, n, dv) else walks
    assert taken <= 1.1 * min(chunks, walks)


@pytest.mark.parametrize("heads,dk,dv,lens,chunks,walks", [
    (128, 64, 16, [130] * 32, 625, 248), (128, 64, 8, [200] * 16, 414, 188), (128, 32, 8, [130] * 16, 159, 78),
    (64, 128, 64, [1000] + [100] * 10, 261, 428), (32, 64, 64, [1000] + [1] * 64, 122, 254), (4, 64, 128, [130] * 2, 23, 36),
    (16, 128, 32, [100] + [1] * 64, 72, 48), (64, 32, 64, [900] * 8, 288, 481), (16, 128, 128, [200], 43, 70)])
def test_linear_attention_of_long_segments(heads, dk, dv, lens, chunks, walks):
    taken = chunks if M._linear_chunks_pay(unlike(lens), heads, dk, dv) else walks
    assert taken <= 1.1 * min(chunks, walks)


@pytest.mark.parametrize("rule,heads,dk,dv,lens,chunks,walks", [
    (M._delta_chunks_pay, 64, 128, 64, [1000] + [100] * 10, 436, 688), (M._delta_chunks_pay, 16, 64, 128, [100] + [1] * 64, 72, 47),
    (M._delta_chunks_pay, 32, 64, 64, [1000] + [1] * 64, 133, 364), (M._ssd_chunks_pay, 16, 128, 128, [300] + [1] * 64, 120, 86),
    (M._ssd_chunks_pay, 128, 16, 32, [3000] + [1] * 64, 187, 436), (M._ssd_chunks_pay, 32, 64, 64, [1000] + [1] * 64, 84, 174)])
def test_prompts_beside_short_segments(rule, heads, dk, dv, lens, chunks, walks):
    assert (chunks if rule(unlike(lens), heads, dk, dv) else walks) <= 1.1 * min(chunks, walks)
