"""CPU checks (compile-only plans) that the larger set of radices changes no length's fate: what
was refused for its prime factors or its size stays refused."""
import pytest

D = pytest.importorskip("dtfft_amd")
P = D.Precision


@pytest.fixture(autouse=True)
def compile_only():
    if D.device_arch().startswith("gfx950"):
        pytest.skip("a GPU is present; compile-only behaviour is exercised on CPU hosts")


def refused(make):
    with pytest.raises(D.DtfftError) as e:
        make()
    assert e.value.code == 602


@pytest.mark.parametrize("n,prec", [(17 * 1000, P.SINGLE), (37 * 512, P.SINGLE), (31 * 200, P.DOUBLE)])
def test_long_lines_with_large_primes_are_refused(n, prec):
    refused(lambda: D.FFTExecutor(1, D.FFTType.C2C, prec, n, n, 1, [n]))
    refused(lambda: D.FFTExecutor(1, D.FFTType.R2C, prec, n, n // 2 + 1, 1, [n], [n], [n // 2 + 1]))


def test_cycle_and_unpack_refuse_large_primes():
    from dtfft_amd import pencil
    refused(lambda: D.Cycle([[34, 16, 16]], P.SINGLE))
    _, recv, _, _ = pencil.forward_exchange(64, 74, 4, 2, 1)
    refused(lambda: D.UnpackFFT((74, 4, 32), recv, P.SINGLE))


@pytest.mark.parametrize("n,prec", [(17 * 600, P.SINGLE), (37 * 138, P.DOUBLE), (61 * 160, P.SINGLE), (59 * 86, P.DOUBLE)])
def test_longest_accepted(n, prec):
    D.FFTExecutor(1, D.FFTType.C2C, prec, n, n, 3, [n])
