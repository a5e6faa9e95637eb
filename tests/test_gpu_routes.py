"""GPU parity of the routes: sizes and alignments at the edges of the one-launch
flat kernels, the matrix-core kernels for wide codes, the rules between them
and the batched kernels' edge tiles, each against the CPU encoder or the scalar
oracle.  Integer work, so the bar is byte equality."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

GUARD = 0x5A


def _carve(dev, arrays, offsets):
    """Device views at the given offsets (mod 16) into one guarded arena each."""
    views, arenas = [], []
    for a, off in zip(arrays, offsets):
        arena = torch.full((a.size + 64,), GUARD, dtype=torch.uint8, device=dev)
        base = (off - arena.data_ptr()) % 16 + 16
        view = arena[base: base + a.size]
        view.copy_(torch.from_numpy(a))
        views.append(view)
        arenas.append((arena, base))
    return views, arenas


def _check(pkg, dev, k, m, n, in_off, out_off, coeff=None, data=None, seed=0):
    rng = np.random.default_rng([k, m, n, seed])
    host = data if data is not None else [rng.integers(0, 256, n, dtype=np.uint8) for _ in range(k)]
    C = oracle.cauchy(k, m) if coeff is None else coeff
    shards, _ = _carve(dev, host, [in_off(j) for j in range(k)])
    outs, arenas = _carve(dev, [np.zeros(n, np.uint8)] * m, [out_off(i) for i in range(m)])
    pkg.matvec(C, shards, out=outs)
    torch.cuda.synchronize()
    want = [np.empty(n, np.uint8) for _ in range(m)]
    oracle.fast_rs_encode(C, host, want)
    for i, ((arena, base), w) in enumerate(zip(arenas, want)):
        got = arena.cpu().numpy()
        assert np.array_equal(got[base: base + n], w), f"RS({k},{m}) n={n} output {i}"
        assert (got[:base] == GUARD).all() and (got[base + n:] == GUARD).all(), \
            f"RS({k},{m}) n={n} output {i}: bytes around it changed"


# unrolled tables in registers / in LDS, the matrix cores with five and more
# outputs, with m <= 4 and k > 16, and the deep codes with their bit matrix in
# registers / in LDS
SHAPES = [(1, 1), (6, 3), (16, 4), (12, 8), (5, 5), (17, 1), (20, 4), (32, 3),
          (13, 6), (24, 8), (31, 9), (32, 16), (4, 12)]


@pytest.mark.parametrize("k,m", SHAPES)
def test_sizes_at_chunk_and_step_edges(pkg, dev, k, m):
    for n in [1, 15, 16, 17, 31, 32, 33, 511, 512, 513, 1024, 2047, 2049, 4096 + 5]:
        _check(pkg, dev, k, m, n, lambda j: 0, lambda i: 0)


@pytest.mark.parametrize("k,m", SHAPES)
@pytest.mark.parametrize("n", [16, 29, 47, 1000, 4133])
def test_every_shard_at_its_own_offset(pkg, dev, k, m, n):
    _check(pkg, dev, k, m, n, lambda j: (5 * j + 3) % 16, lambda i: (7 * i + 1) % 16)
    _check(pkg, dev, k, m, n, lambda j: 9, lambda i: 9)        # one offset for all
    _check(pkg, dev, k, m, n, lambda j: 4 * j % 16, lambda i: 0)   # aligned outputs


@pytest.mark.parametrize("k,m", [(6, 9), (17, 1), (10, 12), (20, 5), (10, 6), (6, 8), (20, 4),
                                 (24, 8), (16, 16)])
def test_both_sides_of_the_table_rule(pkg, dev, k, m):
    """Shards of 2 MiB (matrix cores) and just above (where the tables pay:
    RS(6,9) to RS(6,8))."""
    for n in [2 << 20, (2 << 20) + 16, (2 << 20) + 33]:
        _check(pkg, dev, k, m, n, lambda j: 0, lambda i: 0)
    _check(pkg, dev, k, m, (2 << 20) + 16, lambda j: 4 * j % 16, lambda i: 0)


@pytest.mark.parametrize("k,m", [(17, 1), (20, 2), (17, 3), (13, 5), (32, 2), (6, 9), (10, 12),
                                 (2, 16)])
def test_table_codes_at_any_size_and_alignment(pkg, dev, k, m):
    """table_kernel with both edges, one, or none, and outputs at their own
    offsets: sizes just past the matrix cores' range."""
    n = 4 << 20
    _check(pkg, dev, k, m, n + 16, lambda j: 0, lambda i: 0)
    _check(pkg, dev, k, m, n + 33, lambda j: 0, lambda i: 0)
    _check(pkg, dev, k, m, n + 48, lambda j: 4 * j % 16, lambda i: 4)
    _check(pkg, dev, k, m, n + 2047, lambda j: (5 * j + 3) % 16, lambda i: (7 * i + 1) % 16)


@pytest.mark.parametrize("k,m", [(5, 5), (12, 5), (10, 6), (11, 7), (6, 8)])
def test_any_kernel_with_five_to_eight_outputs(pkg, dev, k, m):
    """Shards just past 2 MiB, where these codes take any_kernel: no edge, a tail,
    both edges, and outputs at offsets of their own."""
    n = 2 << 20
    _check(pkg, dev, k, m, n + 16, lambda j: 0, lambda i: 0)
    _check(pkg, dev, k, m, n + 21, lambda j: 0, lambda i: 0)
    _check(pkg, dev, k, m, n + 33, lambda j: 9, lambda i: 9)
    _check(pkg, dev, k, m, n + 1029, lambda j: (5 * j + 3) % 16, lambda i: (7 * i + 1) % 16)


@pytest.mark.parametrize("k,m,n", [(24, 8, (6 << 20) + 13), (16, 8, (20 << 20) + 13),
                                   (32, 16, (5 << 20) + 13)])
def test_wide_kernel_over_several_steps(pkg, dev, k, m, n):
    """Shards of which every wave of wide_kernel's capped grid codes several
    steps, loading one while it codes another, with both edges."""
    _check(pkg, dev, k, m, n, lambda j: (5 * j + 3) % 16, lambda i: (7 * i + 1) % 16)
    _check(pkg, dev, k, m, n, lambda j: 4, lambda i: 4)


@pytest.mark.parametrize("m", [1, 4, 7, 16])
def test_sums_of_256_ones(pkg, dev, m):
    """32 equal coefficients whose bit matrix has a row of ones: on shards of
    0xFF that row's sum is 256, one more than two bytes per accumulator allow."""
    def full_row(c):
        products = [int(oracle.gf_mul(c, 1 << b)) for b in range(8)]
        return any(all(p >> bit & 1 for p in products) for bit in range(8))
    c = next(c for c in range(1, 256) if full_row(c))
    coeff = np.full((m, 32), c, np.uint8)
    coeff[m // 2:] = oracle.cauchy(32, m)[m // 2:]
    n = 1500
    ones = [np.full(n, 0xFF, np.uint8) for _ in range(32)]
    ones[5][700:] = 3   # both kinds of column next to each other
    for co in (coeff, np.full((m, 32), c, np.uint8)):
        _check(pkg, dev, 32, m, n, lambda j: 0, lambda i: 0, coeff=co, data=ones)


@pytest.mark.parametrize("m", [1, 7, 16])
def test_sums_of_256_ones_batched(pkg, dev, m):
    """The same rows through the batched encode and decode: units of 0xFF, some
    short, some not there."""
    c = next(c for c in range(1, 256)
             if any(all(int(oracle.gf_mul(c, 1 << b)) >> bit & 1 for b in range(8)) for bit in range(8)))
    C = np.full((m, 32), c, np.uint8)
    C[: m // 2] = oracle.cauchy(32, m)[: m // 2]
    k, unit, n = 32, 1040, 5
    ln = np.full((n, k), unit, np.uint32)
    ln[1, 3], ln[2, :] = 517, 1039
    ln[3, 7] = 0
    units = torch.full((n, k, unit), 0xFF, dtype=torch.uint8, device=dev)
    ptr = units.data_ptr() + unit * torch.arange(n * k, dtype=torch.int64, device=dev).view(n, k)
    ptr[3, 7] = 0
    d_len = torch.from_numpy(ln.view(np.int32)).to(dev)
    grid = [[np.full(int(ln[s, j]), 0xFF, np.uint8) if ln[s, j] else None for j in range(k)]
            for s in range(n)]
    want = oracle.encode_batched(C, grid, ln, unit)
    lib, stream = pkg._lib, pkg.codec.stream_handle(torch.cuda.current_stream(), dev)
    out = torch.zeros((2, n, m, unit), dtype=torch.uint8, device=dev)
    o_ptr = out.data_ptr() + unit * torch.arange(2 * n * m, dtype=torch.int64, device=dev).view(2, n, m)
    o_len = torch.full((n, m), unit, dtype=torch.int32, device=dev)
    lib.check(lib.lib().ec_encode_batched(lib.u8ptr(C), k, m, ptr.data_ptr(), d_len.data_ptr(),
                                          o_ptr[0].data_ptr(), n, unit, stream), "ec_encode_batched")
    lib.check(lib.lib().ec_decode_batched(lib.u8ptr(C), k, m, ptr.data_ptr(), d_len.data_ptr(),
                                          o_ptr[1].data_ptr(), o_len.data_ptr(), n, unit, stream),
              "ec_decode_batched")
    torch.cuda.synchronize()
    for got in out:
        assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("k,m", [(6, 3), (10, 6), (24, 8), (20, 4)])
@pytest.mark.parametrize("offset", [0, 5])
def test_output_over_an_input(pkg, dev, k, m, offset):
    """Outputs in place of the first inputs: each byte depends on its own column only."""
    n = 40_007
    rng = np.random.default_rng(k)
    host = [rng.integers(0, 256, n, dtype=np.uint8) for _ in range(k)]
    shards, _ = _carve(dev, host, [offset] * k)
    e = min(k, m)
    C = oracle.cauchy(k, e)
    pkg.matvec(C, shards, out=shards[:e])
    want = [np.empty(n, np.uint8) for _ in range(e)]
    oracle.fast_rs_encode(C, host, want)
    torch.cuda.synchronize()
    for i in range(e):
        assert np.array_equal(shards[i].cpu().numpy(), want[i])


@pytest.mark.parametrize("k,m", [(4, 4), (5, 5), (10, 6), (24, 8), (32, 16)])
def test_output_over_an_input_of_a_few_bytes(pkg, dev, k, m):
    """The same below one chunk, where a lane codes several outputs: none may be
    stored while another is still to be read from what it overwrites."""
    for n in (1, 7, 15):
        rng = np.random.default_rng([k, n])
        host = [rng.integers(0, 256, n, dtype=np.uint8) for _ in range(k)]
        shards, _ = _carve(dev, host, [(3 * j + 1) % 16 for j in range(k)])
        C = oracle.cauchy(k, m)
        pkg.matvec(C, shards, out=shards[:m])
        want = [np.empty(n, np.uint8) for _ in range(m)]
        oracle.fast_rs_encode(C, host, want)
        torch.cuda.synchronize()
        for i in range(m):
            assert np.array_equal(shards[i].cpu().numpy(), want[i]), f"n={n} output {i}"


@pytest.mark.parametrize("k", [1, 2, 5, 16, 17, 32])
def test_xor_any_shards(pkg, dev, k):
    for n in [1, 16, 17, 1023, 1040, 70_001]:
        for off in (lambda j: 0, lambda j: (3 * j + 1) % 16):
            rng = np.random.default_rng([k, n])
            host = [rng.integers(0, 256, n, dtype=np.uint8) for _ in range(k)]
            shards, _ = _carve(dev, host, [off(j) for j in range(k)])
            outs, arenas = _carve(dev, [np.zeros(n, np.uint8)], [off(2)])
            pkg.xor_encode(shards, out=outs[0])
            torch.cuda.synchronize()
            got = arenas[0][0].cpu().numpy()
            base = arenas[0][1]
            assert np.array_equal(got[base: base + n], np.bitwise_xor.reduce(host))
            assert (got[:base] == GUARD).all() and (got[base + n:] == GUARD).all()


def _fill(n, dev, seed):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    return torch.empty(n, dtype=torch.uint8, device=dev).random_(0, 256, generator=g)


def test_unaligned_kernels_past_the_grid_cap(pkg, dev):
    """Shards of 16 GiB + 4141 B at an odd address: more chunks than one pass of
    one-wavefront workgroups covers, with both edges."""
    n = (16 << 30) + 4141
    a, b = _fill(n + 16, dev, 21)[1: 1 + n], _fill(n + 16, dev, 22)[3: 3 + n]
    want = torch.bitwise_xor(a, b)
    x = pkg.xor_encode([a, b])
    assert torch.equal(x, want)
    x = pkg.matvec(np.ones((1, 2), np.uint8), [a, b])[0]
    assert torch.equal(x, want)
    del a, b, want, x
    torch.cuda.empty_cache()


def test_wide_kernel_past_the_grid_cap(pkg, dev):
    """24 shards (one tensor) of 32 GiB + 4101 B through wide_narrow_kernel: more
    than a grid of 256-lane workgroups may hold.  Each row's coefficients add up
    to 1, so every output equals the tensor."""
    n = (32 << 30) + 4101
    a = _fill(n, dev, 23)
    C = np.arange(1, 73, dtype=np.uint8).reshape(3, 24)
    C[:, 0] ^= np.bitwise_xor.reduce(C, axis=1) ^ 1
    outs = pkg.matvec(C, [a] * 24)
    for o in outs:
        assert all(torch.equal(o[i: i + (4 << 30)], a[i: i + (4 << 30)]) for i in range(0, n, 4 << 30))
    del a, outs, o
    torch.cuda.empty_cache()


# ------------------------------------------------------- batched edge tiles --

@pytest.mark.parametrize("k,m,unit", [(4, 2, 1024), (12, 4, 1040), (8, 2, 4096), (6, 3, 16),
                                      (16, 1, 2048), (20, 6, 1024)])
@pytest.mark.parametrize("skew", [0, 1, 6])
def test_units_of_every_length_around_the_chunk(pkg, dev, k, m, unit, skew):
    """Tensors of 1 to 33 bytes and of lengths around a tile, aligned and back
    to back at any byte, through encode, copying encode, decode in place and
    update; bytes between the tensors stay."""
    rng = np.random.default_rng([k, m, unit, skew])
    sizes = list(range(1, 34)) + [unit - 1, unit, unit + 1, unit + 15, 2 * unit + 17, 1007, 1009,
                                  1023, 1025, 1041]
    rng.shuffle(sizes)
    gap = 3 if skew else 0
    starts, at = [], skew
    for sz in sizes:
        starts.append(at)
        at += sz + gap if skew else -(-sz // 16) * 16
    arena = torch.full((at + 64,), GUARD, dtype=torch.uint8, device=dev)
    host = [rng.integers(0, 256, sz, dtype=np.uint8) for sz in sizes]
    tensors = [arena[a: a + sz] for a, sz in zip(starts, sizes)]
    for t, h in zip(tensors, host):
        t.copy_(torch.from_numpy(h))
    lay = pkg.StripeLayout(tensors, k, m, unit)

    def expected(hs):
        grid = []
        for s in range(lay.n_stripes):
            row = []
            for j in range(k):
                u = s * k + j
                t, i = (int(lay.unit_tensor[u]), int(lay.unit_index[u])) if u < lay.n_units \
                    else (-1, 0)
                row.append(hs[t][i * unit: (i + 1) * unit] if t >= 0 else None)
            grid.append(row)
        return oracle.encode_batched(lay.coeff, grid, lay.host_len, unit)

    parity = lay.encode()
    torch.cuda.synchronize()
    want = expected(host)
    assert np.array_equal(parity.cpu().numpy(), want)

    from megatron_lm_amd.checkpoint import GpuSliceCodec
    _, slices = GpuSliceCodec(k, m, unit).encode(tensors)
    for i in range(m):
        assert np.array_equal(slices[k + i], want[:, i].reshape(-1))
    for j in range(k):
        units = np.zeros((lay.n_stripes, unit), np.uint8)
        for s in range(lay.n_stripes):
            u = s * k + j
            if u < lay.n_units:
                piece = host[int(lay.unit_tensor[u])][int(lay.unit_index[u]) * unit:][:unit]
                units[s, : piece.size] = piece
        assert np.array_equal(slices[j], units.reshape(-1))

    before = arena.clone()
    lost = sorted(int(x) for x in rng.choice(k + m, m, replace=False))
    for p in lost:
        if p < k:
            for s in range(lay.n_stripes):
                if s * k + p < lay.n_units:
                    lay.unit_view(s * k + p).fill_(0xEE)
        else:
            parity[:, p - k].fill_(0xEE)
    lay.decode(parity, lost)
    torch.cuda.synchronize()
    assert torch.equal(arena, before), f"lost {lost}"
    assert np.array_equal(parity.cpu().numpy(), want)

    changed = sorted(int(x) for x in rng.choice(lay.n_units, lay.n_units // 2, replace=False))
    old = [lay.unit_view(u).clone() for u in changed]
    for u in changed:
        lay.unit_view(u).bitwise_xor_(0x6B)
    lay.update(parity, changed, old)
    torch.cuda.synchronize()
    now = [t.cpu().numpy() for t in tensors]
    assert np.array_equal(parity.cpu().numpy(), expected(now))


@pytest.mark.parametrize("k,m,unit,n", [(10, 6, 16 << 10, 17 << 20), (20, 2, 64 << 10, 17 << 20),
                                        (24, 8, 4096, 1 << 20), (32, 16, 512, 100_000),
                                        (32, 3, 1536, 50_000)])
def test_batched_wide_routes(pkg, dev, k, m, unit, n):
    """Both sides of the rule between the tables and the matrix cores (16 MiB of
    each position), odd numbers of 512-byte steps, and the deepest code."""
    rng = np.random.default_rng([k, m])
    sizes = [n * k * 3 // 5 + 7, n * k * 2 // 5 + 1, 333]
    flat = torch.randint(0, 256, (sum(sizes) + 64,), dtype=torch.uint8, device=dev,
                         generator=torch.Generator(device=dev).manual_seed(k))
    starts = np.cumsum([0] + [-(-s // 16) * 16 for s in sizes[:-1]])
    tensors = [flat[int(a): int(a) + s] for a, s in zip(starts, sizes)]
    lay = pkg.StripeLayout(tensors, k, m, unit)
    parity = lay.encode()
    # sampled stripes against the scalar oracle
    pick = sorted({0, lay.n_stripes - 1, *(int(x) for x in rng.integers(0, lay.n_stripes, 6))})
    grid, ln = [], []
    for s in pick:
        row = [lay.unit_view(s * k + j).cpu().numpy() if s * k + j < lay.n_units else None
               for j in range(k)]
        grid.append(row)
        ln.append([0 if r is None else r.size for r in row])
    want = oracle.encode_batched(lay.coeff, grid, np.array(ln, np.uint32), unit)
    assert np.array_equal(parity[pick].cpu().numpy(), want)
    # and every stripe back from the parity
    before, par = flat.clone(), parity.clone()
    lost = sorted(int(x) for x in rng.choice(k + m, min(m, 5), replace=False))
    for p in lost:
        if p >= k:
            parity[:, p - k].fill_(1)
    gone = [lay.unit_view(s * k + p) for p in lost if p < k for s in range(lay.n_stripes)
            if s * k + p < lay.n_units]
    torch._foreach_zero_(gone)
    lay.decode(parity, lost)
    assert torch.equal(flat, before) and torch.equal(parity, par)


def test_batched_core_kernel_past_one_grid(pkg, dev):
    """2^24 + 5 stripes of 16-byte units, more than a grid of 256-lane workgroups
    may hold.  The units repeat every 1024 stripes, so each parity unit equals
    that of the first 1024, which the scalar oracle checks."""
    k, m, unit, n, period = 17, 4, 16, (1 << 24) + 5, 1024
    arena = _fill(period * k * unit, dev, 31)
    stripe = torch.arange(n, dtype=torch.int64, device=dev).remainder_(period)
    dptr = torch.empty((n, k), dtype=torch.int64, device=dev)
    for j in range(k):
        torch.add(stripe * (k * unit), arena.data_ptr() + j * unit, out=dptr[:, j])
    dlen = torch.full((n, k), unit, dtype=torch.int32, device=dev)
    parity = torch.zeros((n, m, unit), dtype=torch.uint8, device=dev)
    pptr = parity.data_ptr() + unit * torch.arange(n * m, dtype=torch.int64, device=dev)
    C = oracle.cauchy(k, m)
    lib = pkg._lib
    lib.check(lib.lib().ec_encode_batched(
        lib.u8ptr(C), k, m, dptr.data_ptr(), dlen.data_ptr(), pptr.data_ptr(), n, unit,
        pkg.codec.stream_handle(torch.cuda.current_stream(), torch.device(dev))), "ec_encode_batched")
    torch.cuda.synchronize()
    first = parity[:period]
    units = arena.cpu().numpy().reshape(period, k, unit)
    want = oracle.encode_batched(C, [list(s) for s in units], np.full((period, k), unit, np.uint32), unit)
    assert np.array_equal(first.cpu().numpy(), want)
    for a in range(period, n, 1 << 20):
        b = min(n, a + (1 << 20))
        assert torch.equal(parity[a:b], first[stripe[a:b]])
    del dptr, dlen, pptr, parity
    torch.cuda.empty_cache()
