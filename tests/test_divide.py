"""Divisions of a right-hand side (clode_divide.h): which tokens the program builder replaces, that what it cannot
replace still compiles, and that the quotients by constants are those of IEEE division."""
import os
import subprocess
from fractions import Fraction

import numpy as np
import pytest

import clode_amd as clode
from clode_amd.cpp import clode_cpp_wrapper as w

HEAD = ("void getRHS(const realtype t, const realtype x_[], const realtype p_[], realtype dx_[], realtype aux_[], "
        "const realtype w_[])\n{\n")


def _program(tmp_path, text, precision, compile=False):
    path = tmp_path / "rhs.cl"
    path.write_text(text)
    pi = w.ProblemInfo(str(path), ["x"], ["p"], [], 0)
    sim = w.SimulatorBase(pi, "euler", precision, w.OpenCLResource(), str(tmp_path / "cache"))
    if compile:
        sim.compile()
    s = sim.get_program_string()
    return s[s.index('#line 1 "rhs.cl"'):s.index("clode_rng.h")]


@pytest.mark.parametrize("line, out", [
    ("dx_[0] = a / b;", "dx_[0] = a  *CLODE_DIV*  b;"),
    ("dx_[0] = a/b/c;", "dx_[0] = a *CLODE_DIV* b *CLODE_DIV* c;"),
    ("a /= b;", "a /= b;"),
    ("a = 1; // a / b", "a = 1; // a / b"),
    ("a = b /* x / y */ / c;", "a = b /* x / y */  *CLODE_DIV*  c;"),
    ("a = 1; // a \\\n / b", "a = 1; // a \\\n / b"),
    ("#define F(x) ((x) / \\\n 3.0)\na = F(b) / 2;", "#define F(x) ((x) / \\\n 3.0)\na = F(b)  *CLODE_DIV*  2;"),
    ("const char *s = \"a / \\\" / b\"; char c = '/';", "const char *s = \"a / \\\" / b\"; char c = '/';"),
    ("a = 1'000.0 / b;", "a = 1'000.0  *CLODE_DIV*  b;"),
])
def test_replaced_tokens(tmp_path, line, out):
    assert out in _program(tmp_path, HEAD + line + "\n}\n", False)
    assert line in _program(tmp_path, HEAD + line + "\n}\n", "fp32c")  # divides by reciprocals instead


def test_outside_functions_as_written(tmp_path):
    text = "const int half = 7 / 2;\n" + HEAD + "dx_[0] = p_[0] / half;\n}\n"
    s = _program(tmp_path, text, False)
    assert "half = 7 / 2;" in s and "p_[0]  *CLODE_DIV*  half" in s


# text around divisions that a scanner can take for something else, each a body's lines and its replaced divisions:
# comments that begin on a preprocessor line, with braces, quotes and division signs in them, literals, spliced lines,
# numbers, and text that the program itself can see (a stringified argument), which is left alone
TEXTS = {
    "comment from a define": ("#define TAU 10.0 /* time constant\n  in ms */\n  dx_[0] = -x_[0];\n"
                              "  dx_[0] += p_[0] / TAU; /* drive */", 1),
    "two comments from a define": ("#define K 2 /* a */ /* b\n c\n d */\n dx_[0] = 4.0 / p_[0]; /* c */ aux_[0] = 1;", 1),
    "comment from a pragma": ("#pragma unroll /* all\n */\n for (int i = 0; i < 2; ++i) dx_[0] = x_[i] / 3; /* e */", 1),
    "comment from if and endif": ("#if 1 /* on\n */\n dx_[0] = x_[0] / 3;\n#endif /* off\n } */\n aux_[0] = 1 / p_[0];", 2),
    "braces in the comment": ("#define K 2 /* } } \n { */\n dx_[0] = x_[0] / K;", 1),
    "quotes in the comment": ("#define K 2 /* it's \"so\n */\n dx_[0] = x_[0] / K; /* ' */ aux_[0] = 1 / p_[0];", 2),
    "comment before a directive": ("/* a\n b */ #define K (3 / 2)\n dx_[0] = x_[0] / K;", 1),
    "literal on a directive": ('#define S "/*"\n dx_[0] = x_[0] / 3; /* c */', 1),
    "skipped lines": ("#if 0\n don't / } \n#endif\n dx_[0] = x_[0] / 3;", 1),
    "spliced comment": ("dx_[0] = x_[0] /\\\n/ c\n / 3; /\\\n* a / b *\\\n/ aux_[0] = 1 / p_[0];", 2),
    "spliced string": ('const char *s = "a\\\n/* b"; dx_[0] = x_[0] / 3; /* c */', 1),
    "raw string": ('const char *s = R"x(a " / )" /* )x"; dx_[0] = x_[0] / 3; /* c */', 1),
    "numbers": ("dx_[0] = 1'000'0.0/p_[0] + 0x1p-3/x_[0] + 1.e+3/2;", 3),
    "prefixed literals": ("int c = L'/' + u8'\\'' + '\"'; dx_[0] = c / 3;", 1),
    "digraphs": ("%:define K 2 /* a\n b */\n <% dx_[0] = x_[0] / K; %>", 1),
    "stringified argument": ("#define S(x) #x\n const char *s = S(a / b); dx_[0] = x_[0] / 3;", 0),
    "pasted argument": ("#define S(x) x ## 1\n dx_[0] = x_[0] / 3;", 0),
}


def _tokens(text):
    out = subprocess.run(["g++", "-E", "-P", "-std=c++17", "-w", "-x", "c++", "-"], input=text, text=True,
                         capture_output=True, check=True).stdout
    return "".join(out.split())


@pytest.mark.parametrize("text", list(TEXTS))
def test_same_tokens_as_written(tmp_path, text):
    """After preprocessing, the composed text differs from the written one in the division token alone."""
    body, divisions = TEXTS[text]
    body = HEAD + body + "\n}\n"
    for precision in (True, False):
        s = _program(tmp_path, body, precision)
        s = s[s.index("\n"):s.rindex("#pragma clang force_cuda_host_device end")]
        assert s.count("*CLODE_DIV*") == divisions
        assert _tokens(s).replace("*CLODE_DIV*", "/") == _tokens(body)


# forms of "/" whose operands or results are not plain real numbers; the last cannot go through the operator (its
# left side cannot be copied) and compiles as written
FORMS = {
    "integers": "enum { K = 6 / 2 }; int a[8 / 4]; a[1] = 7 / 2; switch (a[1]) { case 9 / 3: dx_[0] = a[1] / K; }",
    "mixed": "float f = 3.5f; int n = 3; dx_[0] = n / f + f / n + p_[0] / n + 1 / p_[0] + 5 / n;",
    "pointer": "const realtype *q = p_; dx_[0] = x_[0] / *q / -*q;",
    "size": "realtype a[3]; dx_[0] = p_[0] / (sizeof(a) / sizeof(a[0]));",
    "lambda": "auto f = [](auto a, auto b) { return a / b; }; dx_[0] = f(p_[0], 12) + f(7, 2);",
    "constants": "const realtype c = RCONST(1.0) / RCONST(3.0); dx_[0] = c / RCONST(7.0) + 0.0 / 1.0;",
    "vector": "double2 v = make_double2(p_[0], 1.0); dx_[0] = (v / 3.0).x;",
    "own type": "struct R { double v; R(double a) : v(a) {} R(const R &) = delete; double operator/(double d) const "
                "{ return v / d; } }; R r(p_[0]); dx_[0] = r / 3.0;",
}


@pytest.mark.parametrize("precision", [True, False])
@pytest.mark.parametrize("form", list(FORMS))
def test_forms_compile(tmp_path, form, precision):
    _program(tmp_path, HEAD + FORMS[form] + "\n}\n", precision, compile=True)


def test_fallback_is_compiled_once(tmp_path):
    """A text that compiles only as written comes from the cache in the next process, with no attempt at the other."""
    script = tmp_path / "compile.py"
    script.write_text(f"""
import sys
sys.path.insert(0, {os.path.dirname(os.path.dirname(os.path.abspath(__file__)))!r})
import clode_amd as clode
from clode_amd.cpp import clode_cpp_wrapper as w
clode.set_log_level(clode.LogLevel.debug)
pi = w.ProblemInfo({str(tmp_path / "rhs.cl")!r}, ["x"], ["p"], [], 0)
for _ in range(2):
    w.SimulatorBase(pi, "euler", False, w.OpenCLResource(), {str(tmp_path / "cache")!r}).compile()
""")
    (tmp_path / "rhs.cl").write_text(HEAD + FORMS["own type"] + "\n}\n")
    logs = [subprocess.run(["python3", str(script)], capture_output=True, text=True, check=True) for _ in range(2)]
    first, second = (r.stdout + r.stderr for r in logs)
    assert first.count("divisions as written") == 1 and first.count("compiled program") == 1
    assert "build failed" not in second and "compiled program" not in second and second.count("loaded cached code") == 1


# a type whose own division is not that of the real it converts to
OWN = "struct R { double v; double operator/(double d) const { return v * d; } CONVERSION };\n"


def test_own_type_keeps_its_operator(tmp_path, capfd):
    """The operator of an own type is called, not its conversion to double (which here cannot be compiled)."""
    text = OWN.replace("CONVERSION", "template <class T> operator T() const { return typename T::none(0); }")
    level = clode.get_log_level()
    clode.set_log_level(clode.LogLevel.debug)
    try:
        _program(tmp_path, text + HEAD + "R r{p_[0]}; dx_[0] = r / 3.0;\n}\n", False, compile=True)
    finally:
        clode.set_log_level(level)
    out = "".join(capfd.readouterr())
    assert "compiled program" in out and "divisions as written" not in out


@pytest.mark.gpu
def test_own_type_value(tmp_path):
    path = tmp_path / "own.cl"
    path.write_text(OWN.replace("CONVERSION", "operator double() const { return v; }") + HEAD +
                    "R r{p_[0]}; dx_[0] = r / 3.0 + r / x_[0];\n}\n")
    sim = clode.Simulator(src_file=str(path), variables={"x": 2.0}, parameters={"p": 1.0},
                          stepper=clode.Stepper.euler, dt=1.0, t_span=(0.0, 0.5), single_precision=False)
    p = np.arange(1.0, 65.0)
    sim.set_ensemble(parameters={"p": p})
    assert np.array_equal(np.ravel(sim.transient(update_x0=False, fetch_results=True)), 2.0 + p * 3.0 + p * 2.0)


def _quotients(tmp_path, divisor, p, precision):
    """p / divisor as the right-hand side computes it: one Euler step of length 1 from x = 0."""
    path = tmp_path / "q.cl"
    path.write_text(HEAD + f"const realtype c = {divisor};\ndx_[0] = p_[0] / c;\n}}\n")
    sim = clode.Simulator(src_file=str(path), variables={"x": 0.0}, parameters={"p": 1.0},
                          stepper=clode.Stepper.euler, dt=1.0, t_span=(0.0, 0.5), single_precision=precision)
    sim.set_ensemble(variables=np.zeros((p.size, 1)), parameters=p.astype(np.float64)[:, None])
    return np.ravel(sim.transient(update_x0=False, fetch_results=True))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [True, False])
@pytest.mark.parametrize("divisor", ["3", "10", "12.0", "-30", "6", "5300", "524287", "524288.0", "524289", "1000003",
                                     "281474976710655.0", "281474976710657.0", "0.1", "2.5", "8", "1", "-1", "0"])
def test_quotients_by_constants(tmp_path, divisor, precision):
    T, U = (np.float32, np.uint32) if precision else (np.float64, np.uint64)
    r = np.random.default_rng(int(abs(float(divisor))) % 1000)
    c = T(float(divisor))
    tiny = np.finfo(T).tiny
    big = np.finfo(T).max
    anybits = r.integers(0, np.iinfo(U).max, 20000, dtype=U, endpoint=True).view(T)
    # numerators next to c times a middle between two neighbours, where a quotient is hardest to round
    m = (1 + r.random(20000)).astype(T)
    with np.errstate(all="ignore"):
        near = (m * c).astype(T)
        near = (near.view(U) + r.integers(0, 5, near.size).astype(U) - U(2)).view(T)
        special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, tiny, -tiny, big, -big, 1.0, c, -c, c * tiny], T)
        # subnormal numerators and quotients: small multiples of the smallest one, and of it times half the divisor
        unit = np.nextafter(T(0), T(1))
        small = np.arange(-2000, 2001).astype(T) * unit
        edge = ((2 * np.arange(1000) + 1) * (np.abs(c) / T(2))).astype(T) * unit
        p = np.concatenate([anybits, near, special, small, edge])
        want = p / c
        got = _quotients(tmp_path, divisor, p, precision).astype(T)
    # by a whole constant the quotient is formed by multiplication; where the true one is the middle between two
    # subnormals (found in whole numbers of the smallest one), it goes to the neighbour nearer to zero instead of the
    # even one.  Every other quotient is IEEE's, bit for bit
    middle = np.zeros(p.size, bool)
    y = abs(int(c)) if c == np.trunc(c) else 0
    if y and y < (2 ** 19 if precision else 2 ** 48) and y & (y - 1):
        unit = float(np.nextafter(T(0), T(1)))
        for i in np.flatnonzero(np.isfinite(p) & (np.abs(want) <= tiny)):
            x = int(abs(Fraction(float(p[i])) / Fraction(unit)))
            if 2 * x % y == 0 and 2 * x // y % 2:
                middle[i] = True
                want[i] = np.copysign(T(x // y * unit), want[i])
        assert middle.any() == (y % 2 == 0)
    want = want + T(0)  # x = 0 + 1 * (p / c)
    same = (got.view(U) == want.view(U)) | (np.isnan(got) & np.isnan(want))
    assert np.all(same), (p[~same][:5], got[~same][:5], want[~same][:5], middle[~same][:5])


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [True, False, "fp32c"])
def test_comments_from_preprocessor_lines(tmp_path, precision):
    """A model with a comment that begins on a directive gives the states of the same model without comments."""
    got = []
    for text in ("#define TAU 10.0 /* time constant\n in ms */\ndx_[0] = -x_[0];\ndx_[0] += p_[0] / TAU; /* drive */\n",
                 "dx_[0] = -x_[0];\ndx_[0] += p_[0] / 10.0;\n"):
        path = tmp_path / "c.cl"
        path.write_text(HEAD + text + "}\n")
        sim = clode.Simulator(src_file=str(path), variables={"x": 1.0}, parameters={"p": 1.0},
                              stepper=clode.Stepper.rk4, dt=0.01, t_span=(0.0, 2.0), single_precision=precision)
        sim.set_ensemble(parameters={"p": np.linspace(0.5, 9.0, 100)})
        got.append(np.ravel(sim.transient(update_x0=False, fetch_results=True)))
    assert np.array_equal(got[0], got[1])
    t = 2.01  # the first time at or past the span's end
    p = np.linspace(0.5, 9.0, 100) / 10.0
    np.testing.assert_allclose(got[0], p + (1.0 - p) * np.exp(-t), rtol=0.02)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [True, False])
def test_forms_values(tmp_path, precision):
    """The mixed and integer forms give the values of C."""
    path = tmp_path / "q.cl"
    path.write_text(HEAD + "int n = 3; float f = 3.5f;\n"
                    "dx_[0] = p_[0] / n + 7 / 2 + n / f + 1 / p_[0] + 7 / -n + (p_[0] - 5 / 2) / 12 / f;\n}\n")
    T = np.float32 if precision else np.float64
    p = np.linspace(0.5, 9.0, 100).astype(T)
    sim = clode.Simulator(src_file=str(path), variables={"x": 0.0}, parameters={"p": 1.0},
                          stepper=clode.Stepper.euler, dt=1.0, t_span=(0.0, 0.5), single_precision=precision)
    sim.set_ensemble(variables=np.zeros((p.size, 1)), parameters=p.astype(np.float64)[:, None])
    got = np.ravel(sim.transient(update_x0=False, fetch_results=True)).astype(T)
    f = np.float32(3.5)
    want = p / T(3) + T(3) + T(np.float32(3) / f) + T(1) / p + T(-2) + (p - T(2)) / T(12) / T(f)
    np.testing.assert_array_equal(got, want)
