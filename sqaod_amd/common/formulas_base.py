"""Device-independent front end of the formulas modules
(sqaodpy/sqaod/common/formulas_base.py): type fixing, symmetrization and
shape checks, then the device module's function."""
import numpy as np

from . import common


def _as_i8(x):
    return np.ascontiguousarray(np.asarray(x), np.int8)


def _batch(x):
    x = _as_i8(x)
    return x.reshape(1, -1) if x.ndim == 1 else x


def _check_qubo(W):
    if W.ndim != 2 or W.shape[0] != W.shape[1]:
        raise RuntimeError("W must be a square matrix.")


def _check_bipartite(b0, b1, W):
    if W.ndim != 2 or b0.ndim != 1 or b1.ndim != 1 or W.shape != (b1.shape[0], b0.shape[0]):
        raise RuntimeError("Shape mismatch: W must be N1 x N0 for b0[N0], b1[N1].")


# dense graph

# From this size on the device compares W with its transpose, beside the energies:
# a call on 16 float32 states, host / device, is 69 / 85 us at N = 192, 108 / 91 at
# 256, 380 / 158 at 512 (float64 88 / 92, 139 / 101, 598 / 226).
_DEVICE_SYMMETRY_N = 256


def _first_row_symmetric(W):
    # bytes first: a third of the time of the comparison of the numbers
    return W[0].tobytes() == W[:, 0].tobytes() or np.array_equal(W[0], W[:, 0])


def _energies_if_symmetric(cext, cobj, W, x, dtype):
    """E[b] = x_b^T W x_b in one device call, or None where the general path has
    to look at the inputs: W small, not square or not equal to its transpose,
    x of another length.

    A triangular W shows in its first row already (1.3 us at N = 256, 3.8 at
    1000) and does not go to the device for it: a call on 16 float32 states takes
    461 us at N = 256, 4.9 ms at 1000, with the wasted pass 570 us and 5.2 ms."""
    if not isinstance(W, np.ndarray) or W.ndim != 2 or W.shape[0] != W.shape[1] or W.shape[0] < _DEVICE_SYMMETRY_N:
        return None
    if not _first_row_symmetric(W):
        return None
    x = _batch(x)
    if x.ndim != 2 or x.shape[0] == 0 or x.shape[1] != W.shape[0]:
        return None
    E = np.empty((x.shape[0]), dtype)
    return E if cext.dense_graph_batch_calculate_E_if_symmetric(cobj, E, W, x, dtype) else None


def dense_graph_calculate_E(cext, cobj, W, x, dtype):
    W = common.symmetrize(common.fix_type(W, dtype))
    _check_qubo(W)
    x = _as_i8(x)
    if x.shape != (W.shape[0],):
        raise RuntimeError("x must be a vector of length N.")
    E = np.ndarray((1), dtype)
    cext.dense_graph_calculate_E(cobj, E, W, x, dtype)
    return E[0]


def dense_graph_batch_calculate_E(cext, cobj, W, x, dtype):
    W = common.fix_type(W, dtype)
    E = _energies_if_symmetric(cext, cobj, W, x, dtype)
    if E is not None:
        return E
    W = common.symmetrize(W)
    _check_qubo(W)
    x = _batch(x)
    if x.shape[1] != W.shape[0]:
        raise RuntimeError("x rows must have length N.")
    E = np.empty((x.shape[0]), dtype)
    cext.dense_graph_batch_calculate_E(cobj, E, W, x, dtype)
    return E


def dense_graph_calculate_hamiltonian(cext, cobj, W, dtype):
    W = common.symmetrize(common.fix_type(W, dtype))
    _check_qubo(W)
    N = W.shape[0]
    h = np.empty((N), dtype)
    J = np.empty((N, N), dtype)
    c = np.empty((1), dtype)
    cext.dense_graph_calculate_hamiltonian(cobj, h, J, c, W, dtype)
    return h, J, c[0]


def dense_graph_calculate_E_from_spin(cext, cobj, h, J, c, q, dtype):
    h, J = common.fix_type([h, J], dtype)
    J = common.symmetrize(J)
    q = _as_i8(q)
    if h.shape != (J.shape[0],) or q.shape != h.shape:
        raise RuntimeError("Shape mismatch between h, J and q.")
    E = np.ndarray((1), dtype)
    cext.dense_graph_calculate_E_from_spin(cobj, E, h, J, dtype(c), q, dtype)
    return E[0]


def dense_graph_batch_calculate_E_from_spin(cext, cobj, h, J, c, q, dtype):
    h, J = common.fix_type([h, J], dtype)
    J = common.symmetrize(J)
    q = _batch(q)
    if h.shape != (J.shape[0],) or q.shape[1] != h.shape[0]:
        raise RuntimeError("Shape mismatch between h, J and q.")
    E = np.empty((q.shape[0]), dtype)
    cext.dense_graph_batch_calculate_E_from_spin(cobj, E, h, J, dtype(c), q, dtype)
    return E


# bipartite graph

def bipartite_graph_calculate_E(cext, cobj, b0, b1, W, x0, x1, dtype):
    b0, b1, W = common.fix_type([b0, b1, W], dtype)
    _check_bipartite(b0, b1, W)
    x0, x1 = _as_i8(x0), _as_i8(x1)
    E = np.ndarray((1), dtype)
    cext.bipartite_graph_calculate_E(cobj, E, b0, b1, W, x0, x1, dtype)
    return E[0]


def bipartite_graph_batch_calculate_E(cext, cobj, b0, b1, W, x0, x1, dtype):
    b0, b1, W = common.fix_type([b0, b1, W], dtype)
    _check_bipartite(b0, b1, W)
    x0, x1 = _batch(x0), _batch(x1)
    if x0.shape[0] != x1.shape[0]:
        raise RuntimeError("Different batch dims between x0 and x1.")
    E = np.empty((x0.shape[0]), dtype)
    cext.bipartite_graph_batch_calculate_E(cobj, E, b0, b1, W, x0, x1, dtype)
    return E


def bipartite_graph_batch_calculate_E_2d(cext, cobj, b0, b1, W, x0, x1, dtype):
    b0, b1, W = common.fix_type([b0, b1, W], dtype)
    _check_bipartite(b0, b1, W)
    x0, x1 = _batch(x0), _batch(x1)
    E = np.empty((x1.shape[0], x0.shape[0]), dtype)
    cext.bipartite_graph_batch_calculate_E_2d(cobj, E, b0, b1, W, x0, x1, dtype)
    return E


def bipartite_graph_calculate_hamiltonian(cext, cobj, b0, b1, W, dtype):
    b0, b1, W = common.fix_type([b0, b1, W], dtype)
    _check_bipartite(b0, b1, W)
    N0, N1 = W.shape[1], W.shape[0]
    h0 = np.empty((N0), dtype)
    h1 = np.empty((N1), dtype)
    J = np.empty((N1, N0), dtype)
    c = np.empty((1), dtype)
    cext.bipartite_graph_calculate_hamiltonian(cobj, h0, h1, J, c, b0, b1, W, dtype)
    return h0, h1, J, c[0]


def bipartite_graph_calculate_E_from_spin(cext, cobj, h0, h1, J, c, q0, q1, dtype):
    h0, h1, J = common.fix_type([h0, h1, J], dtype)
    _check_bipartite(h0, h1, J)
    E = np.ndarray((1), dtype)
    cext.bipartite_graph_calculate_E_from_spin(cobj, E, h0, h1, J, dtype(c), _as_i8(q0), _as_i8(q1), dtype)
    return E[0]


def bipartite_graph_batch_calculate_E_from_spin(cext, cobj, h0, h1, J, c, q0, q1, dtype):
    h0, h1, J = common.fix_type([h0, h1, J], dtype)
    _check_bipartite(h0, h1, J)
    q0, q1 = _batch(q0), _batch(q1)
    if q0.shape[0] != q1.shape[0]:
        raise RuntimeError("Different batch dims between q0 and q1.")
    E = np.empty((q0.shape[0]), dtype)
    cext.bipartite_graph_batch_calculate_E_from_spin(cobj, E, h0, h1, J, dtype(c), q0, q1, dtype)
    return E
