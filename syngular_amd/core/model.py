"""Tensor-train layers (drop-in for syngular.core, core/model.py:7-226).

``Linear`` holds its weight as a MatrixProductOperator and its forward is
``weight @ inputs`` (core/model.py:201-206): the MPO x MPS apply kernel on
every site, then the reference's ``>> min_bond`` QR truncation, all on the
device.  Extension: a Linear called on a list of states runs the whole batch
in grouped launches (``matmul_batch``), with per-state results equal to
``weight @ x`` one by one.  The reference's console output of ``train`` and
``describe`` is kept; ``train`` adds a random (2,2)x(2,2) bond-4 operator to
every weight as the reference does (core/model.py:33-42).
"""
from __future__ import annotations

import numpy as np
import torch

from .. import _lib, linalg, ops
from ..tensor import MatrixProductOperator, MatrixProductState


# bytes of equally shaped outputs of one site that share a buffer: an output
# that a program keeps holds on to no more than this of the others'
SHARED_BYTES = 1 << 21


def _arena(sizes):
    """One float64 device tensor with a 256-byte aligned sub-buffer per size:
    (tensor, offsets in doubles, addresses)."""
    padded = (sizes + 31) // 32 * 32
    off = np.cumsum(padded) - padded
    t = torch.empty(int(padded.sum()), dtype=torch.float64, device=ops.device())
    return t, off, np.uint64(t.data_ptr()) + (8 * off).astype(np.uint64)


def _outputs(sizes):
    """As _arena for buffers that are results; a list of tensors in place of
    the one, with one a result, where they are too large to share."""
    if 8 * int(sizes.sum()) <= SHARED_BYTES:
        return _arena(sizes)
    dev = ops.device()
    ts = [torch.empty(int(v), dtype=torch.float64, device=dev) for v in sizes]
    return ts, None, np.array([t.data_ptr() for t in ts], dtype=np.uint64)


def _views(t, off, first, count, shape):
    """The tensors of `count` equally shaped neighbours of an arena."""
    l, d, r = (int(v) for v in shape)
    if off is None:
        return [v.view(l, d, r) for v in t[first:first + count]]
    step = (l * d * r + 31) // 32 * 32
    return t.as_strided((count, l, d, r), (step, d * r, r, 1), int(off[first])).unbind(0)


def _state(sites, shape, input_shape, bond_shape, params):
    """A MatrixProductState of device cores of known shapes."""
    mp = MatrixProductState()
    mp.sites, mp.shape, mp.sites_number = sites, shape, len(sites)
    mp.decomposed = True
    mp.parameters_number, mp.real_parameters_number = params, None
    mp.input_shape, mp.bond_shape = input_shape, bond_shape
    return mp


def _gemm_items(it, A, B, C, m, n, k, lda, ta):
    """Fill a grouped GEMM table: C (m x n) = op(A) B, B row-major.  Returns
    (tile, work-groups, flops)."""
    tile = 1 if int((m * n).sum()) >= 256 * 128 * 128 else 0
    bm = 128 if tile else 64
    tn = (n + bm - 1) // bm
    blocks = (m + bm - 1) // bm * tn
    it["A"], it["B"], it["C"], it["m"], it["n"], it["k"] = A, B, C, m, n, k
    it["lda"], it["ldb"], it["ldc"], it["alpha"], it["transA"] = lda, n, n, 1.0, ta
    it["block_start"], it["tiles_n"] = np.cumsum(blocks) - blocks, tn
    return tile, int(blocks.sum()), float((2.0 * m * n * k).sum())


# lists of up to this many states go bond by bond: the array operations of
# matmul_batch cost the same for one state as for fifty (one state of 3 and 6
# cores 261 and 500 us, bond by bond 145 and 311; two 263 and 508, 233 and 519;
# three 270 and 513, 316 and 712)
FEW_STATES = 2


def _matmul_few(weight, states, dims):
    """The launches of matmul_batch with their tables filled bond by bond."""
    n = weight.sites_number
    flat = ops.apply_many([(weight.sites[k], x.sites[k]) for x in states for k in range(n)])
    outs = [MatrixProductState.from_sites(flat[i * n:(i + 1) * n]) for i in range(len(states))]
    if not MatrixProductOperator.COMPRESS:
        return outs
    todo = [i for i, o in enumerate(outs) if dims[i] < min(o.bond_shape)]
    work = {i: outs[i].copy() for i in todo}
    params = {i: 0 for i in todo}
    for k in range(n - 1):
        Ls = [linalg.left_unfold(work[i].sites[k], work[i].shape[k]) for i in todo]
        Rs = [linalg.right_unfold(work[i].sites[k + 1], work[i].shape[k + 1]) for i in todo]
        Qs = ops.qr_many([(L, dims[i]) for L, i in zip(Ls, todo)])
        Ss = [torch.empty((Q.shape[1], L.shape[1]), dtype=torch.float64, device=L.device) for Q, L in zip(Qs, Ls)]
        ops.gemm_many([(Q.t(), L, S, 1.0, 0.0) for Q, L, S in zip(Qs, Ls, Ss)])
        Ws = [torch.empty((S.shape[0], Rm.shape[1]), dtype=torch.float64, device=S.device) for S, Rm in zip(Ss, Rs)]
        ops.gemm_many([(S, Rm, W, 1.0, 0.0) for S, Rm, W in zip(Ss, Rs, Ws)])
        for i, Q, W in zip(todo, Qs, Ws):
            t = work[i]
            t.shape[k] = tuple(t.shape[k][:-1]) + (dims[i],)
            t.shape[k + 1] = (dims[i],) + tuple(t.shape[k + 1][1:])
            t.sites[k] = linalg.reshape(Q, t.shape[k])
            t.sites[k + 1] = linalg.reshape(W, t.shape[k + 1])
            params[i] += t.sites[k].numel()
    for i in todo:
        work[i].parameters_number = params[i] + work[i].sites[-1].numel()
        outs[i] = work[i]
    return outs


def matmul_batch(weight, states):
    """[weight @ x for x in states] (tensor/matrix_product_operator.py:175-192
    per state) in grouped launches: one MPO x MPS apply launch for every site
    of every state, then the QR truncation to each state's min bond
    (tensor/matrix_product_state.py:432-468), bond by bond, with one QR launch
    and two GEMM launches per bond over all the states that need it.  Every
    buffer's address is known before the first launch, so the tables of all
    launches are filled by array operations over the states and go to the
    device in one copy (64 states of 6 cores spent 12 ms on the host in one
    tensor and one table row at a time, against 0.5 ms of kernels).  States
    whose site count differs from the operator's or whose shapes do not chain,
    or a non-default matmul / rounding mode, go through ``weight @ x`` one by
    one."""
    states = list(states)
    n = weight.sites_number
    if (MatrixProductOperator.MATMUL_MODE != "standard" or MatrixProductState.ROUNDING != "qr"
            or any(x.sites_number != n for x in states)):
        return [weight @ x for x in states]
    if not states:
        return []
    dims = [min(min(weight.bond_shape), min(x.bond_shape)) for x in states]
    if len(states) <= FEW_STATES:
        return _matmul_few(weight, states, dims)
    # states of equal shapes next to each other
    members = {}
    for i, x in enumerate(states):
        members.setdefault((dims[i], *(s.shape for s in x.sites)), []).append(i)
    keys = list(members)
    if any(len(s) != 3 for key in keys for s in key[1:]):
        return [weight @ x for x in states]
    X = np.array([key[1:] for key in keys], dtype=np.int64)               # group, site, (l, d, r)
    D = np.array([key[0] for key in keys], dtype=np.int64)
    O = np.array([s.shape for s in weight.sites], dtype=np.int64)         # site, (l, in, out, r)
    P = np.stack([X[:, :, 0] * O[:, 0], np.broadcast_to(O[:, 2], X.shape[:2]), X[:, :, 2] * O[:, 3]], axis=2)
    cut = D < P[:, :-1, 2].min(axis=1) if MatrixProductOperator.COMPRESS else np.zeros(len(keys), bool)
    rows = P[:, :, 0] * P[:, :, 1]                                        # rows of the left unfoldings
    rows[:, 1:] = np.where(cut[:, None], D[:, None] * P[:, 1:, 1], rows[:, 1:])
    if ((X[:, :, 1] != O[:, 1]).any() or P.min() <= 0 or (cut & (D <= 0)).any()
            or (P[cut, :-1, 2] != P[cut, 1:, 0]).any() or (rows[cut, :-1] < D[cut, None]).any()):
        return [weight @ x for x in states]

    order = [i for g in members.values() for i in g]
    count = np.array([len(g) for g in members.values()])
    first = np.cumsum(count) - count
    rep = np.repeat(np.arange(len(keys)), count)
    hold = [[s.contiguous() for s in states[i].sites] for i in order]     # inputs, alive until the launch
    ws = [w.contiguous() for w in weight.sites]
    new = _arena if cut.all() else _outputs     # product cores that are results
    cores = [new(P[rep, k].prod(axis=1)) for k in range(n)]

    # the tables, one after the other in one buffer
    J = len(order)
    todo = cut[rep]
    T = int(todo.sum())
    ap, qr = np.dtype(_lib.APPLY_ITEM), np.dtype(_lib.QR_ITEM)
    ge = np.dtype(_lib.GEMM_ITEM)
    nbytes = J * n * ap.itemsize + (n - 1) * T * (qr.itemsize + 2 * ge.itemsize)
    table, at = np.zeros(nbytes, dtype=np.uint8), 0

    def take(dtype, cnt):
        nonlocal at
        o, at = at, at + cnt * dtype.itemsize
        return o, table[o:at].view(dtype)

    _, it = take(ap, J * n)
    it = it.reshape(J, n)
    it["x"] = [[s.data_ptr() for s in h] for h in hold]
    it["o"] = [w.data_ptr() for w in ws]
    it["p"] = np.stack([c[2] for c in cores], axis=1)
    it["chil"], it["din"], it["chir"] = X[rep, :, 0], X[rep, :, 1], X[rep, :, 2]
    it["dl"], it["dout"], it["dr"] = O[:, 0], O[:, 2], O[:, 3]
    nel = P[rep].prod(axis=2)
    blocks = ((nel + _lib.APPLY_BLOCK - 1) // _lib.APPLY_BLOCK).reshape(-1)
    it["block_start"] = (np.cumsum(blocks) - blocks).reshape(J, n)
    apply_bytes = 8.0 * float(nel.sum() + X[rep].prod(axis=2).sum() + J * O.prod(axis=1).sum())

    steps, done, carry = [], [], []
    if T:
        sel = rep[todo]                                                   # group of each truncated state
        Dt = D[sel]
        core = cores[0][2][todo]
        for k in range(n - 1):
            m, r = rows[sel, k], P[sel, k, 2]
            cols = P[sel, k + 1, 1] * P[sel, k + 1, 2]
            nb = np.minimum(r, Dt)
            Q, S = _outputs(m * Dt), _arena(Dt * r)
            W = (_outputs if k == n - 2 else _arena)(Dt * cols)
            work, tau = _arena(m * nb), _arena(nb)
            oq, it = take(qr, T)
            it["a"], it["rs"], it["cs"], it["m"], it["n"], it["keep"] = core, r, 1, m, r, Dt
            it["q"], it["ldq"], it["work"], it["tau"] = Q[2], Dt, work[2], tau[2]
            o1, it = take(ge, T)
            g1 = _gemm_items(it, Q[2], core, S[2], Dt, r, m, Dt, 1)
            o2, it = take(ge, T)
            g2 = _gemm_items(it, S[2], cores[k + 1][2][todo], W[2], Dt, cols, r, r, 0)
            steps.append((oq, o1, g1, o2, g2))
            done.append(Q)
            carry.append((S, W, work, tau))
            core = W[2]

    dev = ops._device_table(table)
    base, stream = dev.data_ptr(), ops._stream()
    if ops._profiling[0]:
        _lib.call("syn_prof_note_flops", apply_bytes)
    _lib.call("syn_mpo_apply_f64", base, J * n, int(blocks.sum()), stream)
    for oq, o1, g1, o2, g2 in steps:
        _lib.call("syn_qr_f64", base + oq, T, stream)
        for o, (tile, total, flops) in ((o1, g1), (o2, g2)):
            if ops._profiling[0]:
                _lib.call("syn_prof_note_flops", flops)
            _lib.call("syn_gemm_f64", base + o, T, total, tile, stream)

    outs = [None] * J
    at = 0                                                                # first truncated state of the group
    for g, key in enumerate(keys):
        c = int(count[g])
        input_shape, bond_shape = tuple(P[g, :, 1].tolist()), tuple(P[g, :-1, 2].tolist())
        shape = [tuple(v) for v in P[g].tolist()]
        if cut[g]:
            d = int(D[g])
            shape = [(shape[k][0] if k == 0 else d, shape[k][1], d if k < n - 1 else shape[k][2]) for k in range(n)]
            held = [(*done[k][:2], at) for k in range(n - 1)] + [(*carry[-1][1][:2], at)]
            at += c
        else:
            held = [(*cores[k][:2], int(first[g])) for k in range(n)]
        params = sum(l * d * r for l, d, r in shape)
        per_site = [_views(t, off, f, c, sh) for (t, off, f), sh in zip(held, shape)]
        for i, sites in zip(members[key], zip(*per_site)):
            outs[i] = _state(list(sites), list(shape), input_shape, bond_shape, params)
    return outs


class Model:
    # core/model.py:7-82

    def __init__(self, layers):
        self.layers = layers

    def predict(self, inputs):
        values = inputs
        for layer in self.layers:
            values = layer(values)
        return values

    def feed_forward(self, sample):
        values = sample
        for layer in self.layers:
            values = layer(values)
        return values

    def build(self):
        for layer in self.layers:
            if not layer.is_built:
                layer.build(None)
                layer.is_built = True

    def train(self, x, y, batchsize=32, epochs=1, verbose=1):
        if verbose:
            print("[START] Training ")
        for e in range(epochs):
            if verbose:
                print(f"Epoch {str(e + 1)} : ")
            for layer in self.layers:
                for weight in layer.trainable_tensor_weights:
                    weight["weight"] += MatrixProductOperator.random((2, 2), (2, 2), (4,))
        if verbose:
            print("[END] Training ")

    def draw(self):
        return "".join(layer.draw() for layer in self.layers)

    def describe(self):
        strict_layer = ["output"]
        params = params_fictive = layers_num = 0
        rule = "-" * 111
        for layer in self.layers:
            info = layer.describe()
            layers_num += 1
            params += info["param"]
            params_fictive += info["fictive-param"]
            print(rule)
            if info["type"] not in strict_layer:
                saved = info["fictive-param"] - info["param"]
                print(f"|  Layer [{info['type']}] -> {info['name']} \t Parameters: {info['param']} \t "
                      f"Saved: {saved} (compression {round(saved / info['fictive-param'], 4) * 100}%)")
            else:
                print(f"|  Layer [{info['type']}] ->  {info['name']} \t ")
            print(rule)
        print("=" * 111)
        print(f"| \t Total number of layers : {layers_num}")
        print(f"| \t Total number of parameters : {params} (v.s {params_fictive})")
        print(f"| \t Total compression factor : {round((params_fictive - params) / params_fictive, 4) * 100}%")
        print("=" * 111)


class Layer:
    # core/model.py:84-160

    def __init__(self, name):
        self.name = name
        self.trainable_tensor_weights = []
        self.trainable_tensor_bias = []
        self.is_built = False

    def __call__(self, inputs):
        input_shape = inputs.shape if not isinstance(inputs, (list, tuple)) else None
        if not self.is_built:
            self.build(input_shape)
            self.is_built = True

    def build(self, input_shape):
        pass

    def draw(self):
        out = ""
        for weight in self.trainable_tensor_weights:
            mp = weight["weight"]
            out += "\t" + "|   " * mp.sites_number + "\n"
            out += "\t" + ("O---" * (mp.sites_number - 1)) + "O" + "\n"
            out += "\t" + "|   " * mp.sites_number + "\n"
        return out

    def describe(self):
        total = sum(w["weight"].parameters_number for w in self.trainable_tensor_weights)
        total += sum(b["bias"].parameters_number for b in self.trainable_tensor_bias)
        true = sum(w["weight"].real_parameters_number for w in self.trainable_tensor_weights)
        true += sum(b["bias"].real_parameters_number for b in self.trainable_tensor_bias)
        return {"param": total, "fictive-param": true, "name": self.name, "type": self.type}

    def add_weight(self, input_shape, output_shape, bond_shape, name=None, initializer="normal"):
        if name is None:
            name = f"weight_{np.random.randint(0, 999999)}"
        weight = MatrixProductOperator.random(input_shape, output_shape, bond_shape)
        self.trainable_tensor_weights.append({"name": name, "weight": weight})

    def add_bias(self, size, name=None, initializer="normal"):
        pass


class Linear(Layer):
    # core/model.py:162-206

    def __init__(self, input_units, output_units, core=1, bond=None, bias_initializer="normal",
                 weights_initializer="normal", activation="relu", name="linear"):
        super().__init__(name)
        self.input_units = input_units
        self.output_units = output_units
        self.core = core
        self.bond_dimension = bond
        self.input_core_dim = round(self.input_units ** (1 / self.core))
        self.output_core_dim = round(self.output_units ** (1 / self.core))
        self._input_shape = (self.input_core_dim,) * self.core
        self._output_shape = (self.output_core_dim,) * self.core
        self._bond_shape = (self.bond_dimension,) * (self.core - 1)
        self.bias_initializer = bias_initializer
        self.weights_initializer = weights_initializer
        self.activation = activation
        self.type = "linear"

    def build(self, input_shape):
        if self.weights_initializer == "normal":
            self.add_weight(self._input_shape, self._output_shape, bond_shape=self._bond_shape, name="weight",
                            initializer="normal")
        else:
            self.trainable_tensor_weights.append({"name": "", "weight": self.weights_initializer})

    def __call__(self, inputs):
        super().__call__(inputs)
        weight = self.trainable_tensor_weights[0]["weight"]
        if isinstance(inputs, (list, tuple)):
            return matmul_batch(weight, inputs)
        return weight @ inputs


class Output(Layer):
    # core/model.py:208-218

    def __init__(self, output_shape, name="output"):
        super().__init__(name)
        self.output_shape = output_shape
        self.type = "output"

    def __call__(self, inputs):
        if isinstance(inputs, (list, tuple)):
            return [x.to_tensor().reshape(self.output_shape) for x in inputs]
        return inputs.to_tensor().reshape(self.output_shape)
