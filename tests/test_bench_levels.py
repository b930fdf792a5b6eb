"""bench.py's prices and kernel names of the CD 2D launches of several levels:
a plan that steps two per launch (variant code 22) takes the same kernel, and
the same byte model, as one that steps eight (88)."""
import bench

E = 4
N = 1000 * 100
NS = (1000, 100)
STRIP = bench._strip_cells(NS, 0) * 2 * E


def test_two_levels_are_priced_as_several():
    nt, S = 501, 50
    kl = (nt - 1) // S
    last, rep = nt - kl * S, kl * S
    for n in (2, 3, 8):
        launches = kl * -(-S // n) + -(-last // n)
        replays = kl * -(-S // n)
        fwd, adj = (bench.alg_bytes("cd2d", NS, 0, E, [nt], S, (11, 11 * n))[k] for k in (0, 1))
        assert fwd == ((launches + replays) * (5 * E * N + STRIP) + (last + rep) * E * N, launches + replays)
        assert adj == (launches * (7 * E * N + STRIP) + nt * E * N, launches)


def test_kernel_names_follow_the_levels():
    assert bench.kernel_names("cd2d", [2, 11])[0] == "cd2d_step_kernel<float, 2> (forward)"
    for code in (22, 55, 88):
        assert bench.kernel_names("cd2d", [20, code]) == ("cd2d_stepn_kernel<float, 8, 8, false> (forward)",
                                                          "cd2d_stepn_kernel<float, 2, 16, true> (adjoint)")
