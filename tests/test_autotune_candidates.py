"""The autotuner times no two parameter sets that the library runs alike."""
import autotune


def acts_as(p):
    return p.tile, p.micro, p.big, min(max(p.small, p.tile ** 2 // 2), p.tile ** 2 + 1)


def test_candidates_are_distinct_and_complete():
    got = autotune.candidates()
    assert len({acts_as(p) for p in got}) == len(got)
    want = {acts_as(autotune.Params(t, m, s, b)) for t in autotune.TILES for m in autotune.MICROS
            for s in autotune.SMALLS for b in autotune.BIGS}
    assert {acts_as(p) for p in got} == want
    # 8: half, whole, none; 16: half, 192, none; 32: half, whole
    assert [sum(p.tile == t for p in got) for t in (8, 16, 32)] == [3 * 18, 3 * 18, 2 * 18]
