"""``set_alpha`` on operators of other classes (host, no GPU)."""
import pgj


class _OneArgument:
    """An operator whose unscaled Green apply takes the residual alone."""

    def green_precond(self, r):
        return -r


def test_unscaled_green_takes_the_residual_alone():
    op = pgj.set_alpha(_OneArgument(), 0)
    assert op.apply_precond(3) == -3
