// butterfly.hpp -- forward DFT butterflies of radix 2 .. 17 on registers, the
// in-register part of the line kernels' stages: X_k = sum_m v_m e^{-2 pi i m k / R},
// natural order in and out.  The line kernels run every transform forward
// (an inverse one exchanges real and imaginary parts of its inputs and
// outputs), so the direction is no operand here and every rotation by -i is
// a register renaming.
//
// Composite radices with coprime factors (6, 10, 12, 14, 15) are prime-factor
// transforms: no twiddles between their two dimensions, only index maps.
#pragma once

#include "device.hpp"

namespace rfh {
namespace dev {

template <typename T>
__device__ __forceinline__ C2<T> mul_mi(C2<T> a) {  // a * -i
  return {a.y, -a.x};
}

// cos / sin of 2 pi q / P for q = 1 .. (P - 1) / 2
template <int P>
struct PrimeRoots;
template <>
struct PrimeRoots<7> {
  static constexpr double c[3] = {0.6234898018587335305250048840042398, -0.222520933956314404288902564496794,
                                  -0.900968867902419126236102319507445};
  static constexpr double s[3] = {0.7818314824680298087084445266740578, 0.9749279121818236070181316829939312,
                                  0.4338837391175581204757683328483588};
};
template <>
struct PrimeRoots<11> {
  static constexpr double c[5] = {0.8412535328311811688618116489193677, 0.4154150130018864255292741492296232,
                                  -0.142314838273285140443792668616369, -0.654860733945285064056925072466293,
                                  -0.959492973614497389890368057066327};
  static constexpr double s[5] = {0.5406408174555975821076359543186917, 0.9096319953545183714117153830790285,
                                  0.9898214418809327323760920377767188, 0.7557495743542582837740358439723444,
                                  0.2817325568414296977114179153466169};
};
template <>
struct PrimeRoots<13> {
  static constexpr double c[6] = {0.8854560256532098959003755220150989, 0.5680647467311558025118075591275166,
                                  0.1205366802553230533490676874525436, -0.354604887042535625969637892600018,
                                  -0.748510748171101098634630599701351, -0.970941817426052027156982276293789};
  static constexpr double s[6] = {0.4647231720437685456560153351331048, 0.8229838658936563945796174234393820,
                                  0.9927088740980539928007516494925202, 0.9350162426854148234397845998378307,
                                  0.6631226582407952023767854926667663, 0.2393156642875577671487537262602119};
};
template <>
struct PrimeRoots<17> {
  static constexpr double c[8] = {0.9324722294043558045731158918215634, 0.7390089172206591159245343098726481,
                                  0.4457383557765382673964575493794869, 0.0922683594633019952396511071545065,
                                  -0.273662990072082863539077935436813, -0.602634636379256389178588154986840,
                                  -0.850217135729614152134143922949352, -0.982973099683901778281948844855198};
  static constexpr double s[8] = {0.3612416661871529487447145961837002, 0.6736956436465572117126919124256946,
                                  0.8951632913550622220670164997537855, 0.9957341762950345218711911789054818,
                                  0.9618256431728190704087962907315186, 0.7980172272802395033328051127962614,
                                  0.5264321628773558002446077991406996, 0.1837495178165703315744088396207276};
};

template <int R>
struct Bfly;

template <int R, typename T>
__device__ __forceinline__ void bfly(C2<T> *v) {
  Bfly<R>::run(v);
}

template <>
struct Bfly<2> {
  template <typename T>
  static __device__ __forceinline__ void run(C2<T> *v) {
    const C2<T> a = v[0];
    v[0] = a + v[1];
    v[1] = a - v[1];
  }
};

template <>
struct Bfly<3> {
  template <typename T>
  static __device__ __forceinline__ void run(C2<T> *v) {
    const T s = T(0.866025403784438646763723170752936183);
    const C2<T> t = v[1] + v[2], d = v[1] - v[2];
    const C2<T> a = {v[0].x - T(0.5) * t.x, v[0].y - T(0.5) * t.y};
    v[0] = v[0] + t;
    v[1] = {a.x + s * d.y, a.y - s * d.x};
    v[2] = {a.x - s * d.y, a.y + s * d.x};
  }
};

template <>
struct Bfly<4> {
  template <typename T>
  static __device__ __forceinline__ void run(C2<T> *v) {
    const C2<T> t0 = v[0] + v[2], t1 = v[0] - v[2], t2 = v[1] + v[3];
    const C2<T> t3 = mul_mi(v[1] - v[3]);
    v[0] = t0 + t2;
    v[2] = t0 - t2;
    v[1] = t1 + t3;
    v[3] = t1 - t3;
  }
};

template <>
struct Bfly<5> {
  template <typename T>
  static __device__ __forceinline__ void run(C2<T> *v) {
    const T c1 = T(0.309016994374947424102293417182819059);
    const T c2 = T(-0.809016994374947424102293417182819059);
    const T s1 = T(0.951056516295153572116439333379382143);
    const T s2 = T(0.587785252292473129168705954639072769);
    const C2<T> t1 = v[1] + v[4], t2 = v[2] + v[3], d1 = v[1] - v[4], d2 = v[2] - v[3];
    const C2<T> a1 = v[0] + c1 * t1 + c2 * t2, a2 = v[0] + c2 * t1 + c1 * t2;
    const C2<T> b1 = mul_mi(s1 * d1 + s2 * d2), b2 = mul_mi(s2 * d1 - s1 * d2);
    v[0] = v[0] + t1 + t2;
    v[1] = a1 + b1;
    v[4] = a1 - b1;
    v[2] = a2 + b2;
    v[3] = a2 - b2;
  }
};

template <>
struct Bfly<8> {
  template <typename T>
  static __device__ __forceinline__ void run(C2<T> *v) {
    C2<T> e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    bfly<4>(e);
    bfly<4>(o);
    const T s = T(0.707106781186547524400844362104849039);
    const C2<T> o1 = {s * (o[1].x + o[1].y), s * (o[1].y - o[1].x)};
    const C2<T> o2 = mul_mi(o[2]);
    const C2<T> o3 = {s * (o[3].y - o[3].x), -s * (o[3].x + o[3].y)};
    v[0] = e[0] + o[0];
    v[4] = e[0] - o[0];
    v[1] = e[1] + o1;
    v[5] = e[1] - o1;
    v[2] = e[2] + o2;
    v[6] = e[2] - o2;
    v[3] = e[3] + o3;
    v[7] = e[3] - o3;
  }
};

// 3 x 3: DFT3 over x[n2], x[n2 + 3], x[n2 + 6], twiddle W9^(n2 k1), DFT3 over n2
template <>
struct Bfly<9> {
  template <typename T>
  static __device__ __forceinline__ void run(C2<T> *v) {
    const C2<T> w1 = {T(0.766044443118978035202392650555416674), T(-0.642787609686539326322643409907263433)};
    const C2<T> w2 = {T(0.173648177666930348851716626769314796), T(-0.984807753012208059366743024589523014)};
    const C2<T> w4 = {T(-0.93969262078590838405410927732473147), T(-0.342020143325668733044099614682259581)};
    C2<T> a[3] = {v[0], v[3], v[6]}, b[3] = {v[1], v[4], v[7]}, c[3] = {v[2], v[5], v[8]};
    bfly<3>(a);
    bfly<3>(b);
    bfly<3>(c);
    b[1] = cmul(b[1], w1);
    b[2] = cmul(b[2], w2);
    c[1] = cmul(c[1], w2);
    c[2] = cmul(c[2], w4);
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
      C2<T> t[3] = {a[k1], b[k1], c[k1]};
      bfly<3>(t);
      v[k1] = t[0];
      v[k1 + 3] = t[1];
      v[k1 + 6] = t[2];
    }
  }
};

// 4 x 4: DFT4 over x[4 n1 + n2], twiddle W16^(n2 k1), DFT4 over n2
template <>
struct Bfly<16> {
  template <typename T>
  static __device__ __forceinline__ void run(C2<T> *v) {
    const T c1 = T(0.923879532511286756128183189396788933);
    const T s1 = T(0.382683432365089771728459984030398866);
    const T r = T(0.707106781186547524400844362104849039);
    C2<T> a[4][4];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < 4; ++n1) a[n2][n1] = v[4 * n1 + n2];
      bfly<4>(a[n2]);
    }
    a[1][1] = cmul(a[1][1], C2<T>{c1, -s1});
    a[1][2] = {r * (a[1][2].x + a[1][2].y), r * (a[1][2].y - a[1][2].x)};
    a[1][3] = cmul(a[1][3], C2<T>{s1, -c1});
    a[2][1] = {r * (a[2][1].x + a[2][1].y), r * (a[2][1].y - a[2][1].x)};
    a[2][2] = mul_mi(a[2][2]);
    a[2][3] = {r * (a[2][3].y - a[2][3].x), -r * (a[2][3].x + a[2][3].y)};
    a[3][1] = cmul(a[3][1], C2<T>{s1, -c1});
    a[3][2] = {r * (a[3][2].y - a[3][2].x), -r * (a[3][2].x + a[3][2].y)};
    a[3][3] = cmul(a[3][3], C2<T>{-c1, s1});
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
      C2<T> t[4] = {a[0][k1], a[1][k1], a[2][k1], a[3][k1]};
      bfly<4>(t);
#pragma unroll
      for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = t[k2];
    }
  }
};

// Odd prime P through the symmetric pairs x_m +- x_{P-m}.
template <int P>
struct BflyPrime {
  template <typename T>
  static __device__ __forceinline__ void run(C2<T> *v) {
    constexpr int H = (P - 1) / 2;
    C2<T> t[H], d[H];
    const C2<T> x0 = v[0];
#pragma unroll
    for (int m = 1; m <= H; ++m) {
      t[m - 1] = v[m] + v[P - m];
      d[m - 1] = v[m] - v[P - m];
    }
    C2<T> sum = x0;
#pragma unroll
    for (int m = 0; m < H; ++m) sum = sum + t[m];
    v[0] = sum;
#pragma unroll
    for (int k = 1; k <= H; ++k) {
      C2<T> a = x0, b = {T(0), T(0)};
#pragma unroll
      for (int m = 1; m <= H; ++m) {
        const int q = (m * k) % P;
        const T c = T(PrimeRoots<P>::c[(q <= H ? q : P - q) - 1]);
        const T s = q <= H ? T(PrimeRoots<P>::s[q - 1]) : T(-PrimeRoots<P>::s[P - q - 1]);
        a = a + c * t[m - 1];
        b = b + s * d[m - 1];
      }
      v[k] = {a.x + b.y, a.y - b.x};
      v[P - k] = {a.x - b.y, a.y + b.x};
    }
  }
};
template <>
struct Bfly<7> : BflyPrime<7> {};
template <>
struct Bfly<11> : BflyPrime<11> {};
template <>
struct Bfly<13> : BflyPrime<13> {};
template <>
struct Bfly<17> : BflyPrime<17> {};

// Coprime factors A x B: input n = (B n1 + A n2) mod AB, output k with
// k = k1 mod A, k = k2 mod B, no twiddles (W_AB^(nk) = W_A^(n1 k1) W_B^(n2 k2)).
constexpr int crt(int A, int B, int k1, int k2) {
  int k = k1;
  while (k % B != k2) k += A;
  return k;
}
template <int A, int B>
struct BflyPfa {
  template <typename T>
  static __device__ __forceinline__ void run(C2<T> *v) {
    C2<T> a[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) a[n2][n1] = v[(B * n1 + A * n2) % (A * B)];
      bfly<A>(a[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      C2<T> t[B];
#pragma unroll
      for (int n2 = 0; n2 < B; ++n2) t[n2] = a[n2][k1];
      bfly<B>(t);
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) v[crt(A, B, k1, k2)] = t[k2];
    }
  }
};
template <>
struct Bfly<6> : BflyPfa<3, 2> {};
template <>
struct Bfly<10> : BflyPfa<5, 2> {};
template <>
struct Bfly<12> : BflyPfa<4, 3> {};
template <>
struct Bfly<14> : BflyPfa<7, 2> {};
template <>
struct Bfly<15> : BflyPfa<5, 3> {};

}  // namespace dev
}  // namespace rfh
