"""A closed box of mirrors with the light outside and a narrow view straight at
one wall: without roulette its paths run to and fro up to the bounce limit."""
import numpy as np

import yune_amd as Y


def mirror_box():
    s = Y.gen_cornell()
    rows = []
    for axis in range(3):
        for side in (-1.0, 1.0):
            c = np.zeros((4, 3))
            c[:, axis] = side
            c[:, (axis + 1) % 3] = (-1, 1, 1, -1)
            c[:, (axis + 2) % 3] = (-1, -1, 1, 1)
            n = np.zeros(3)
            n[axis] = -side
            rows += [(c[0], c[1], c[2], n), (c[0], c[2], c[3], n)]
    s.tris = np.zeros(len(rows), dtype=Y.TRI_DTYPE)
    for t, (a, b, c, n) in zip(s.tris, rows):
        for k, v in (("v1", a), ("v2", b), ("v3", c)):
            t[k] = (*v, 1)
        for k in ("vn1", "vn2", "vn3"):
            t[k] = (*n, 0)
    s.mats = s.mats[:1].copy()
    s.mats["is_specular"] = 1
    s.mats["is_transmissive"] = 0
    s.mats["ke"] = 0
    s.mats["ke"][0, 0] = 1e-3       # so that a path's sample counts its bounces
    s.light = Y.light_quad((50, 50, 50), (0, -1, 0), (1, 1, 1), (0.1, 0, 0), (0, 0, 0.1))
    s.cam = Y.camera((1, 0, 0), (0, 1, 0), (0, 0, -1), (0.6, -0.5, 0.3), 1e-5)   # clear of the walls' diagonals
    s.nodes = None
    return s
