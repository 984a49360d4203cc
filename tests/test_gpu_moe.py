"""GPU parity for the MoE-routed SG path: routing and per-expert lists exact
against the oracle, gathered rows byte-exact, RMSNorm within a bf16 tolerance
of the fp32 oracle."""
import numpy as np
import pytest

import gfd_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    assert gfd_amd.device_count() > 0, "no GPU visible to libgfd_amd.so"
    assert gfd_amd.lib().gfd_set_device(0) == 0


class Moe:
    def __init__(self, tokens, experts, dim, stride_factor=2):
        self.T, self.E, self.dim = tokens, experts, dim
        self.row_bytes = dim * 2
        self.stride = stride_factor * self.row_bytes
        self.values = oracle.moe_token_values(tokens, dim)
        self.host = gfd_amd.HostBuffer(tokens * self.stride)
        self.host.array[:] = oracle.GAP_BYTE
        rows = self.host.array.reshape(tokens, self.stride)
        rows[:, :self.row_bytes] = self.values.view(np.uint8).reshape(tokens, self.row_bytes)
        self.logits = oracle.moe_logits(tokens, experts)
        self.top2 = oracle.moe_top2(self.logits)
        self.offsets, self.row_token = oracle.moe_lists(self.top2, experts)
        self.weight = oracle.moe_weight(dim)
        self.d_logits = gfd_amd.DeviceBuffer(self.logits.nbytes)
        self.d_logits.upload(self.logits)
        self.d_top2 = gfd_amd.DeviceBuffer(tokens * 2 * 4)
        self.d_offsets = gfd_amd.DeviceBuffer((experts + 1) * 4)
        self.d_rows = gfd_amd.DeviceBuffer(tokens * 2 * 4)
        self.d_weight = gfd_amd.DeviceBuffer(dim * 2)
        self.d_weight.upload(self.weight)
        n = 2 * tokens
        self.d_dst = gfd_amd.DeviceBuffer(n * self.row_bytes + 4096)
        self.d_out = gfd_amd.DeviceBuffer(n * self.row_bytes + 4096)
        self.d_err = gfd_amd.DeviceBuffer(4)

    def route(self):
        gfd_amd.moe_route(self.d_logits.ptr, self.T, self.E, self.d_top2.ptr, self.d_offsets.ptr, self.d_rows.ptr)
        gfd_amd.synchronize()

    def gather(self, with_norm, eps=1e-6, blocks=0):
        self.d_dst.fill(0xCD)
        self.d_out.fill(0xCD)
        self.d_err.fill(0)
        gfd_amd.sg_gather_rmsnorm(self.host.ptr, self.stride, self.T, self.d_rows.ptr, 2 * self.T, self.row_bytes,
                                  self.d_dst.ptr, self.d_out.ptr if with_norm else None,
                                  self.d_weight.ptr, eps, blocks, self.d_err.ptr)
        gfd_amd.synchronize()
        assert int(self.d_err.download().view(np.int32)[0]) == 0

    def expected_rows(self):
        return self.values[self.row_token]


CASES = [(4096, 64, 7168), (64, 8, 512), (300, 5, 1024), (1000, 16, 2048)]


@pytest.mark.parametrize("T,E,dim", CASES)
def test_route_and_lists_exact(T, E, dim):
    m = Moe(T, E, dim)
    m.route()
    top2 = m.d_top2.download().view(np.int32).reshape(T, 2)
    assert (top2 == m.top2).all()
    assert (m.d_offsets.download().view(np.int32) == m.offsets).all()
    assert (m.d_rows.download().view(np.int32) == m.row_token).all()


@pytest.mark.parametrize("T,E,dim", CASES)
def test_gather_rows_byte_exact(T, E, dim):
    m = Moe(T, E, dim)
    m.route()
    m.gather(with_norm=False)
    n = 2 * T
    got = m.d_dst.download()
    assert (got[:n * m.row_bytes].view(np.uint16).reshape(n, dim) == m.expected_rows()).all()
    assert (got[n * m.row_bytes:] == 0xCD).all()
    assert (m.d_out.download() == 0xCD).all()  # pure transfer writes no norm output


@pytest.mark.parametrize("T,E,dim", CASES)
def test_gather_with_rmsnorm(T, E, dim):
    m = Moe(T, E, dim)
    m.route()
    eps = 1e-6
    m.gather(with_norm=True, eps=eps)
    n = 2 * T
    rows = m.expected_rows()
    got_rows = m.d_dst.download()[:n * m.row_bytes].view(np.uint16).reshape(n, dim)
    assert (got_rows == rows).all()
    ref = oracle.rmsnorm_rows(oracle.bf16_to_f32(rows), oracle.bf16_to_f32(m.weight), eps)
    got = oracle.bf16_to_f32(m.d_out.download()[:n * m.row_bytes].view(np.uint16).reshape(n, dim))
    # bf16 output: within one bf16 ulp of the fp32 reference (relative 2^-7),
    # and almost every element rounds to the same bf16 value.
    assert np.all(np.abs(got - ref) <= np.abs(ref) * 2.0 ** -7 + 1e-6)
    same = np.mean(oracle.f32_to_bf16(ref) == oracle.f32_to_bf16(got))
    assert same > 0.99
    assert (m.d_out.download()[n * m.row_bytes:] == 0xCD).all()


def test_gather_rejects_bad_row_bytes():
    m = Moe(64, 8, 512)
    with pytest.raises(gfd_amd.GfdError):
        gfd_amd.sg_gather_rmsnorm(m.host.ptr, m.stride, m.T, m.d_rows.ptr, 2 * m.T, 1000, m.d_dst.ptr, None,
                                  None, 1e-6, 0, m.d_err.ptr)


def test_gather_flags_out_of_range_token():
    m = Moe(64, 8, 512)
    bad = np.arange(2 * m.T, dtype=np.int32) % m.T
    bad[5] = m.T + 3
    m.d_rows.upload(bad)
    m.d_err.fill(0)
    gfd_amd.sg_gather_rmsnorm(m.host.ptr, m.stride, m.T, m.d_rows.ptr, 2 * m.T, m.row_bytes, m.d_dst.ptr, None,
                              None, 1e-6, 4, m.d_err.ptr)
    gfd_amd.synchronize()
    assert int(m.d_err.download().view(np.int32)[0]) & 4


# Tokens around the one-launch limit (512), the waves' groups (64) and the
# runs kept in registers (8192); experts around the 16 lanes of a token.
@pytest.mark.parametrize("T", [1, 15, 64, 65, 511, 512, 513, 1025, 8191, 8192, 8193, 20001])
@pytest.mark.parametrize("E", [2, 3, 16, 17, 63, 64])
def test_route_edges(T, E):
    """top2, offsets and row lists exact, with ties (lower expert first), -inf
    logits, and guards behind every output."""
    print("route T=%d E=%d" % (T, E), flush=True)
    rng = np.random.default_rng(T * 100 + E)
    logits = rng.integers(-3, 4, (T, E)).astype(np.float32)  # many ties
    logits[rng.random((T, E)) < 0.2] = -np.inf
    logits[:, rng.permutation(E)[:2]] = (4.0, 5.0)  # two finite ones in every row
    logits[: T // 2] += rng.standard_normal((T // 2, E), dtype=np.float32)
    top2 = oracle.moe_top2(logits)
    offsets, rows = oracle.moe_lists(top2, E)
    d = gfd_amd.DeviceBuffer(logits.nbytes)
    d.upload(logits)
    outs = [gfd_amd.DeviceBuffer(4 * n + 64) for n in (2 * T, E + 1, 2 * T)]
    for o in outs:
        o.fill(0xCD)
    gfd_amd.moe_route(d.ptr, T, E, outs[0].ptr, outs[1].ptr, outs[2].ptr)
    gfd_amd.synchronize()
    got = [o.download() for o in outs]
    for g, n in zip(got, (2 * T, E + 1, 2 * T)):
        assert (g[4 * n:] == 0xCD).all()
    assert (got[0][:8 * T].view(np.int32) == top2.reshape(-1)).all()
    assert (got[1][:4 * (E + 1)].view(np.int32) == offsets).all()
    k = len(rows)
    assert (got[2][:4 * k].view(np.int32) == rows).all()


@pytest.mark.parametrize("T", [300, 5000])
def test_route_of_nan_rows_stays_in_range(T):
    """A row that holds NaN still routes to experts that exist."""
    E = 5
    logits = np.random.default_rng(T).standard_normal((T, E), dtype=np.float32)
    logits[np.random.default_rng(T + 1).random((T, E)) < 0.4] = np.nan
    d, t2, off, rows = [gfd_amd.DeviceBuffer(n) for n in (logits.nbytes, 8 * T, 4 * (E + 1), 8 * T)]
    d.upload(logits)
    rows.fill(0)
    gfd_amd.moe_route(d.ptr, T, E, t2.ptr, off.ptr, rows.ptr)
    gfd_amd.synchronize()
    top2 = t2.download().view(np.int32)
    assert (top2 >= 0).all() and (top2 < E).all()
    clean = ~np.isnan(logits).any(1)
    assert (top2.reshape(T, 2)[clean] == oracle.moe_top2(logits[clean])).all()
    o = off.download().view(np.int32)
    assert o[0] == 0 and o[E] == 2 * T and (np.diff(o) >= 0).all()
    r = rows.download().view(np.int32)
    assert (r >= 0).all() and (r < T).all()


@pytest.mark.parametrize("T", [300, 5000])
@pytest.mark.parametrize("E", [2, 5, 64])
def test_route_of_rows_without_two_finite_logits(T, E):
    """Rows of NaN, -inf and +inf: the two experts are distinct, so that every
    row of the lists is written; a NaN ranks behind everything, ties go to the
    lower expert."""
    print("route of NaN and infinite rows T=%d E=%d" % (T, E), flush=True)
    rng = np.random.default_rng(T + E)
    logits = rng.standard_normal((T, E), dtype=np.float32)
    logits[rng.random((T, E)) < 0.4] = np.nan
    one = rng.integers(0, E, T)
    for kind, (fill, at) in enumerate([(np.nan, None), (np.nan, 1.0), (-np.inf, None), (-np.inf, 1.0), (np.nan, -np.inf),
                                       (-np.inf, np.nan), (np.inf, np.nan), (-np.inf, np.inf), (np.inf, None)]):
        t = np.arange(kind, T, 12)
        logits[t] = fill
        if at is not None:
            logits[t, np.where(t % 24 == kind, one[t], 0)] = at  # at any expert, and at expert 0
    top2 = oracle.moe_top2(logits)
    offsets, rows = oracle.moe_lists(top2, E)
    d = gfd_amd.DeviceBuffer(logits.nbytes)
    d.upload(logits)
    outs = [gfd_amd.DeviceBuffer(4 * n) for n in (2 * T, E + 1, 2 * T)]
    for o in outs:
        o.fill(0xCD)
    gfd_amd.moe_route(d.ptr, T, E, outs[0].ptr, outs[1].ptr, outs[2].ptr)
    gfd_amd.synchronize()
    got = [o.download().view(np.int32) for o in outs]
    assert (top2[:, 0] != top2[:, 1]).all()
    assert (got[0] == top2.reshape(-1)).all()
    assert (got[1] == offsets).all()
    assert (got[2] == rows).all()
