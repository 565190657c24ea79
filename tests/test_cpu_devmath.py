"""The kernels' FP64 primitives (dev_math.h) on the host against 80-bit
arithmetic: their largest error in units of the last place stays at or below
that of the general functions whose place they take, which the file's header
states.  The header is compiled as C++ with the hardware's approximations in
their documented accuracy (23 bits) and its inline fused multiply-add as
fma ()."""
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
KERNELS = os.path.join(HERE, "..", "marx_amd", "csrc", "kernels")

SHIM = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>
#define __device__
#define __host__
#define __forceinline__ inline
using std::copysign; using std::fabs; using std::fma; using std::fmax; using std::rint;
static double coarse (double x)
{
   uint64_t u; memcpy (&u, &x, 8); u &= ~((1ull << 29) - 1); memcpy (&x, &u, 8); return x;
}
static double mantissa (double x) { int e; return std::frexp (x, &e); }
static int exponent (double x) { int e; std::frexp (x, &e); return e; }
static int __double2loint (double x) { uint64_t u; memcpy (&u, &x, 8); return (int) (uint32_t) u; }
#define __builtin_amdgcn_rcp(x) coarse (1.0 / (x))
#define __builtin_amdgcn_rsq(x) coarse (1.0 / std::sqrt (x))
#define __builtin_amdgcn_frexp_mant(x) mantissa (x)
#define __builtin_amdgcn_frexp_exp(x) exponent (x)
#define __builtin_amdgcn_div_fixup(q, b, a) ((std::isfinite (q) && (q) != 0.0) ? (q) : (a) / (b))
#define __builtin_amdgcn_bitop3_b32(a, b, c, d) ((a) ^ (b) ^ (c))
"""

MAIN = r"""
using namespace mxg;
static double polar_scale (double g) %s

struct Worst
{
   double ulps = 0;
   void operator() (double got, long double want)
   {
      const double a = std::fabs ((double) want);
      const double e = (double) (fabsl (got - want) / (std::nextafter (a, INFINITY) - a));
      if (!(e <= ulps)) ulps = e;       // a NaN stays
   }
};

int main ()
{
   std::mt19937_64 gen (11);
   std::uniform_real_distribution<double> uniform (0.0, 1.0);
   Worst lg, polar, rs, sq, dv, sn[4], cs[4];
   double turn = 0.0;
   const double top[4] = {0.785, 100.0, 6.0e4, 1048576.0};
   for (int i = 0; i < (1 << 18); i++)
     {
        const double u = uniform (gen), v = uniform (gen), x = std::exp (-80.0 * u * u * u);
        if (u == 0.0) continue;
        lg (log_n (u), logl (u));
        lg (log_n (x), logl (x));
        const double y = 1.0 / x;
        lg (log_n (y), logl (y));
        polar (polar_scale (u), sqrtl (-2.0L * logl (u) / u));
        rs (rsqrt_n (x), 1.0L / sqrtl (x));
        sq (sqrt_n (x), sqrtl (x));
        dv (div_n (v, 1.0 + 9.0 * u), (long double) v / (1.0 + 9.0 * u));
        double s, c;
        for (int k = 0; k < 4; k++)
          {
             const double t = (2.0 * v - 1.0) * top[k];
             sincos_r (t, s, c);
             sn[k] (s, sinl (t));
             cs[k] (c, cosl (t));
             sn[k] (sin_r (t), sinl (t));
          }
        sincos_turn (u, s, c);
        const long double a = 6.283185307179586476925286766559L * u;
        turn = std::fmax (turn, (double) fmaxl (fabsl (s - sinl (a)), fabsl (c - cosl (a))));
        // to 2^50 with an absolute error below 4e-16
        const double big = std::ldexp (1.0 + u, 20 + (int) (29.0 * v));
        sincos_r (big, s, c);
        if (!(std::fabs (s * s + c * c - 1.0) < 1e-15)) turn = NAN;
        if (!(std::fabs (s - std::sin (big)) < 4e-16) || !(std::fabs (c - std::cos (big)) < 4e-16)) turn = NAN;
     }
   printf ("log %%g polar %%g rsqrt %%g sqrt %%g div %%g turn %%g log(1) %%g sqrt(0) %%g", lg.ulps, polar.ulps, rs.ulps, sq.ulps, dv.ulps,
           turn, log_n (1.0), sqrt_n (0.0));
   for (int k = 0; k < 4; k++) printf (" sin%%d %%g cos%%d %%g", k, sn[k].ulps, k, cs[k].ulps);
   return 0;
}
"""


def _function_body(text, name):
    """The braces of the function `name` in the source text."""
    i = text.index("{", text.index(name + " ("))
    depth, j = 0, i
    while True:
        depth += {"{": 1, "}": -1}.get(text[j], 0)
        j += 1
        if depth == 0:
            return text[i:j]


@pytest.fixture(scope="module")
def worst(tmp_path_factory):
    d = tmp_path_factory.mktemp("devmath")
    with open(os.path.join(KERNELS, "dev_math.h")) as f:
        header = f.read()
    header, n = re.subn(r'asm \("v_fma_f64[^;]*;', "d = fma (a, b, c);", header)
    assert n == 1
    header = header.replace("#include <hip/hip_runtime.h>", "").replace("#pragma once", "")
    with open(os.path.join(KERNELS, "dev_common.h")) as f:
        polar = _function_body(f.read(), "polar_scale")
    src = d / "devmath.cpp"
    src.write_text(SHIM + header + MAIN % polar)
    # the kernels contract nothing that is not written as fma
    subprocess.run(["g++", "-O2", "-std=gnu++17", "-ffp-contract=off", "-mfma", "-o", str(d / "devmath"), str(src)],
                   check=True)
    out = subprocess.run([str(d / "devmath")], check=True, capture_output=True, text=True).stdout.split()
    return dict(zip(out[::2], map(float, out[1::2])))


@pytest.mark.parametrize("name,bar", [("div", 0.502), ("sqrt", 0.502), ("rsqrt", 1.0), ("log", 0.63), ("polar", 0.95)]
                         + [(f"{f}{k}", 0.77) for f in ("sin", "cos") for k in range(4)])
def test_largest_error_in_units_of_the_last_place(worst, name, bar):
    assert worst[name] <= bar


def test_whole_turns_and_end_points(worst):
    assert worst["turn"] <= 1.5e-16
    assert worst["log(1)"] == 0.0 and worst["sqrt(0)"] == 0.0
