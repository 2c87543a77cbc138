// Roots of unity of the odd radices, as compile-time constants for the
// butterflies of sgpe_mixed.h. Plain C++ (no HIP).
//
// Written out rather than summed up from series at compile time: in double
// arithmetic a series with its rounded argument came out one or two units in
// the last place off for most entries (cos(2 pi / 3) = -0.49999999999999994). Such
// an error is the same at every butterfly of every pass, so it adds up over a
// run: two steps of 208 x 130, complex128, ended 1.12 times as far from a
// 64-bit transform's result as with exact constants.
#pragma once

namespace sgpe {

// {cos, sin} of 2 pi m / R, m = 1 .. (R - 1) / 2, to 22 decimals (the compiler
// rounds them to the nearest double).
template <int R> struct MixHalf;
template <> struct MixHalf<3> {
  static constexpr double v[1][2] = {{-0.5, 0.8660254037844386467637}};
};
template <> struct MixHalf<5> {
  static constexpr double v[2][2] = {{0.3090169943749474241023, 0.9510565162951535721164},
                                     {-0.8090169943749474241023, 0.5877852522924731291687}};
};
template <> struct MixHalf<7> {
  static constexpr double v[3][2] = {{0.6234898018587335305250, 0.7818314824680298087084},
                                     {-0.2225209339563144042889, 0.9749279121818236070181},
                                     {-0.9009688679024191262361, 0.4338837391175581204758}};
};
template <> struct MixHalf<9> {
  static constexpr double v[4][2] = {{0.7660444431189780352024, 0.6427876096865393263226},
                                     {0.1736481776669303488517, 0.9848077530122080593667},
                                     {-0.5, 0.8660254037844386467637},
                                     {-0.9396926207859083840541, 0.3420201433256687330441}};
};
template <> struct MixHalf<11> {
  static constexpr double v[5][2] = {{0.8412535328311811688618, 0.5406408174555975821076},
                                     {0.4154150130018864255293, 0.9096319953545183714117},
                                     {-0.1423148382732851404438, 0.9898214418809327323761},
                                     {-0.6548607339452850640569, 0.7557495743542582837740},
                                     {-0.9594929736144973898904, 0.2817325568414296977114}};
};
template <> struct MixHalf<13> {
  static constexpr double v[6][2] = {{0.8854560256532098959004, 0.4647231720437685456560},
                                     {0.5680647467311558025118, 0.8229838658936563945796},
                                     {0.1205366802553230533491, 0.9927088740980539928008},
                                     {-0.3546048870425356259696, 0.9350162426854148234398},
                                     {-0.7485107481711010986346, 0.6631226582407952023768},
                                     {-0.9709418174260520271570, 0.2393156642875577671488}};
};

// cos and sin of 2 pi m / R for 0 <= m < R.
template <int R> struct MixUnit {
  double c[R], s[R];
  constexpr MixUnit() : c{}, s{} {
    c[0] = 1.0;
    for (int m = 1; m <= R / 2; ++m) {
      c[m] = c[R - m] = MixHalf<R>::v[m - 1][0];
      s[m] = MixHalf<R>::v[m - 1][1];
      s[R - m] = -s[m];
    }
  }
};
template <int R> struct MixUnitTable { static constexpr MixUnit<R> u{}; };

}  // namespace sgpe
