"""Rounding of the sphere products against exactly summed matrix elements."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WIDE = np.longdouble


def element_by_element(c, x):
    """the row's elements dealt to four partial sums in turn, each term one fused multiply-add in double"""
    parts = [np.zeros(x.shape[1]) for _ in range(4)]
    for i in range(c.size):
        parts[i % 4] = (WIDE(c[i]) * x[i].astype(WIDE) + parts[i % 4]).astype(np.float64)
    return (parts[0] + parts[2]) + (parts[1] + parts[3])


# few rows on eight lanes (338 and 8512 rows), many on one lane (246448)
@pytest.mark.parametrize("n,lz_max,k,nbr_rows", [(6, 15, 8, 338), (6, 15, 1, 338), (8, 21, 1, 400), (10, 27, 1, 150),
                                                 (10, 27, 4, 100)])
def test_products_round_no_more_than_their_elements_one_by_one(arch, n, lz_max, k, nbr_rows):
    """The diagonal elements of a row are summed before they meet x.  That must not cost accuracy: the error of
    the product stays below that of the elements added one by one in double."""
    from diagham_amd import capi
    p = capi.Problem.sphere(arch, n, 0, lz_max, capi.coulomb_pseudopotentials(lz_max))
    X = np.random.default_rng(7).standard_normal((p.dim, k))
    Y = p.hv(X.reshape(-1), k).reshape(p.dim, k)
    got = plain = 0.0
    for r in np.unique(np.linspace(0, p.dim - 1, nbr_rows).astype(int)):
        t, c = p.row_elements(int(r))
        exact = (c.astype(WIDE)[:, None] * X[t].astype(WIDE)).sum(0)
        got += float(((Y[r].astype(WIDE) - exact) ** 2).sum())
        plain += float(((element_by_element(c, X[t]).astype(WIDE) - exact) ** 2).sum())
    p.close()
    assert got <= plain, (np.sqrt(got), np.sqrt(plain))
