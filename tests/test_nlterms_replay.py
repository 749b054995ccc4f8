"""Host replay of nlterms_kernel's transforms (tbl_rhs.hip): the in-place
passes, their digit-reversed order and the even/odd packing against the direct
sums of the transform pair, for every size; LDS slots in bounds."""
import numpy as np
import pytest


def radix(L):
    return 8 if L % 64 == 32 or L >= 128 else 2 if L == 8 else 4


def passes(M, FR):
    L, out = M, []
    while L > FR:
        out.append(L)
        L //= radix(L)
    assert L == FR
    return out


def run_pass(x, N, L, R, up):
    M, J = len(x), L // R
    F = np.exp(-2j * np.pi * np.outer(np.arange(R), np.arange(R)) / R)
    tw = np.exp(-2j * np.pi * np.arange(N) / N)
    for b in range(M // R):
        j = b % J
        at = b // J * L + j + np.arange(R) * J
        w = tw[j * np.arange(R) * (N // L)]
        x[at] = F @ (x[at] * w) if up else (F @ x[at]) * w


@pytest.mark.parametrize("N", [4, 8, 16, 32, 64, 128, 256, 512, 1024])
def test_transform_pair(N):
    M = N // 2
    FR = 4 if M >= 4 else 2
    rng = np.random.default_rng(N)
    K = max(1, M - (N % 3))
    a, b = (rng.normal(size=K) + 1j * rng.normal(size=K) for _ in range(2))
    tw = np.exp(-2j * np.pi * np.arange(N) / N)
    n = np.arange(N)

    def down(c):
        c = np.concatenate([c, np.zeros(M + 1 - K)])
        z = np.zeros(M, complex)
        for m1 in range(max(1, M // 2)):
            m2 = M - m1 if m1 else M // 2
            if m1:
                p, q = 0.5 * c[m1], 0.5 * c[m2]
                z[m1] = p + q.conj() + 1j * (p - q.conj()) * tw[m1]
                z[m2] = q + p.conj() + 1j * (q - p.conj()) * tw[m2]
            else:
                z[0] = (c[0].real + 0.5 * c[0].imag) + 1j * (c[0].real - 0.5 * c[0].imag)
                q = 0.5 * c[m2]
                z[m2] = q + q.conj() + 1j * (q - q.conj()) * tw[m2]
        for L in passes(M, FR):
            run_pass(z, N, L, radix(L), False)
        run_pass(z, N, FR, FR, False)
        return z

    def values(c):
        v = c[0].real + 0.5 * c[0].imag * (-1.0) ** n
        for m in range(1, K):
            v = v + (c[m] * np.exp(-2j * np.pi * m * n / N)).real
        return v

    # the digit-reversed values are those of the direct sum
    za, zb = down(a), down(b)
    va, vb = values(a), values(b)
    assert np.allclose(np.sort(za.real), np.sort(va[::2]), atol=1e-11)
    assert np.allclose(np.sort(za.imag), np.sort(va[1::2]), atol=1e-11)
    y = za.real * zb.real - 1j * za.imag * zb.imag
    run_pass(y, N, FR, FR, True)
    for L in reversed(passes(M, FR)):
        run_pass(y, N, L, radix(L), True)
    w = y.conj()
    got = np.zeros(M, complex)
    for m1 in range(max(1, M // 2)):
        m2 = M - m1 if m1 else M // 2
        u, v = w[m1], w[m2]
        if m1:
            e, d = 0.5 * (u + v.conj()), 0.5 * (u - v.conj())
            o = -1j * d * tw[m1].conj()
            got[m1], got[m2] = 2 / N * (e + o), 2 / N * (e - o).conj()
        else:
            got[0], got[m2] = (u.real + u.imag) / N, 2 / N * v
    ref = np.array([(2.0 if m else 1.0) / N * np.sum(va * vb * np.exp(2j * np.pi * m * n / N)) for m in range(M)])
    ref[0] = ref[0].real
    assert np.allclose(got, ref, atol=1e-11 * np.max(np.abs(ref)) + 1e-13)


@pytest.mark.parametrize("N", [4, 8, 16, 32, 64, 128, 256, 512, 1024])
def test_slots_and_items(N):
    M, P = N // 2, 1024 // N
    slot = np.arange(M) + (np.arange(M) >> 3)
    seq = (slot[-1] + 1) * P
    assert len(set(slot)) == M and (slot[-1] * P + P - 1) < seq
    assert 16 * (6 * seq + N) <= 160 * 1024
    # 256 threads: every mode of every point once (mode 0 pairs with M / 2)
    t = np.arange(256)
    p, m1 = t % P, t // P
    m2 = np.where(m1 > 0, M - m1, M // 2)
    seen = np.zeros((M, P), int)
    np.add.at(seen, (m1, p), 1)
    np.add.at(seen, (m2, p), 1)
    assert np.all(seen == 1)
    FR = 4 if M >= 4 else 2
    for b in range(M // FR):
        assert np.array_equal(slot[FR * b:FR * b + FR], slot[FR * b] + np.arange(FR))
    for L in passes(M, FR):
        R = radix(L)
        j = np.arange(M // R) % (L // R)
        assert (j[:, None] * np.arange(R) * (N // L)).max() < N
