"""Grids that reach every form of the strip kernel: (lx, ly, the block's x
columns and sites, a term in two phases).  That each grid takes the named form
is checked on the CPU (test_strip_shape.py)."""

FORMS = [
    (24, 24, (2, 4), True), (37, 23, (2, 4), False), (2, 20, (2, 4), True),
    (11, 85, (2, 5), True), (340, 5, (2, 5), True), (37, 64, (2, 5), False),
    (9, 72, (2, 6), True), (11, 95, (2, 6), False), (61, 42, (2, 6), True),
    (48, 48, (2, 8), True), (13, 85, (2, 8), False), (64, 64, (2, 8), True),
    (13, 100, (2, 10), True), (15, 87, (2, 10), False), (97, 99, (2, 10), False), (100, 100, (2, 10), True),
    (3, 840, (1, 20), True), (3, 803, (1, 20), False), (85, 31, (1, 20), False),
    (36, 36, (4, 4), True), (44, 44, (4, 4), True),
]
