"""The sort's scratch holds what the sort in use keeps: a second copy of the records only where they are first grouped
by x plane, a count matrix of keys or of planes, whichever is counted.  Sizes from the library, whose host
code runs against a HIP runtime that runs nothing."""
import pytest

from test_lds_attributes import lines_of

CUS = 256

PROGRAM = """
def scatter(n, np, stencil, tile=None):
    t = None if tile is None else C.cast((C.c_int * 3)(1, tile, 0), C.c_void_p)
    need = C.c_size_t()
    ok(lib.pk_scatter_workspace_size(n, np, stencil, t, C.byref(need)))
    return need.value
def slot(n, np, nb, tile):
    plan, need = C.c_void_p(), []
    ok(lib.pk_plan_create(n, C.byref(plan)))
    for jobs in (1, 2):
        s = C.c_size_t()
        ok(lib.pk_batch_workspace_size(plan, jobs, np, nb, C.cast((C.c_int * 3)(1, tile, 0), C.c_void_p), C.byref(s)))
        need.append(s.value)
    return need[1] - need[0]
"""


def bound(n, np, ncls, tile):
    """(largest scratch that the sort of this geometry needs, its kind)"""
    ntiles = n * (n // tile)
    nkeys = ntiles * ncls + 1
    kind = "keys" if nkeys <= 4000 else "mixed" if nkeys <= (160 * 1024 - 16384) // 4 else "planes"
    columns = n + 1 if kind == "planes" else nkeys
    if kind == "mixed":
        columns += n + 1
    nblk = min(CUS, -(-np // 4096))
    records = 16 * np * (1 if kind == "keys" else 2)
    fixed = 16 * 256 + 32 * CUS   # alignment of the parts; statistics and weight sums
    return records + 4 * (nblk + 1) * columns + 8 * nkeys + 16 * ntiles + 4 * (n + 2) + fixed, kind


# (side, rows per tile, classes of the stencil, kind of sort)
CASES = [(32, 32, 2, "keys"), (128, 32, 3, "keys"), (256, 32, 2, "mixed"), (512, 32, 3, "mixed"), (768, 16, 2, "planes"),
         (1024, 16, 2, "planes"), (1024, 16, 3, "planes"), (4096, 4, 2, "planes")]


@pytest.mark.parametrize("np", [1000, 30_000_000])
def test_scratch_is_what_the_sort_uses(np, tmp_path):
    calls = "".join(f"print(scatter({n}, {np}, {2 if ncls == 3 else 1}, {tile}))\n" for n, tile, ncls, _ in CASES)
    for (n, tile, ncls, kind), got in zip(CASES, lines_of(PROGRAM + calls, tmp_path)):
        most, k = bound(n, np, ncls, tile)
        assert k == kind
        assert int(got) <= most, (n, tile, ncls, int(got), most)


def test_a_batch_slot_holds_the_scratch_of_every_job(tmp_path):
    # 512 with 16 rows: TSC jobs count planes, CIC jobs keys beside them (the larger matrix)
    n, tile, np, nb = 512, 16, 2_000_000, 100
    calls = f"print(slot({n}, {np}, {nb}, {tile}))\nprint(scatter({n}, {np}, 1, {tile}))\nprint(scatter({n}, {np}, 2, {tile}))\n"
    got, cic, tsc = map(int, lines_of(PROGRAM + calls, tmp_path))
    spectrum = (n // 2 + 1) * n * n * 8
    assert bound(n, np, 2, tile)[1] == "mixed" and bound(n, np, 3, tile)[1] == "planes"
    assert got >= spectrum + max(cic, tsc)
