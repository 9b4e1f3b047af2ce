// Walks every LDS access of the standard scheme's marches (kernels_std.hip) over
// all waves, rows and lanes, and counts those outside the plane of their level.
#include <cstdio>

#include "../hicar_amd/csrc/std_planes.hpp"

using namespace icaradv;

static int bad = 0;

template <class P>
void in_plane(const char *what, int H, int V, int RW, int r, int c)
{
    const int a = P::at(r, c);
    if (a >= 0 && a < P::SIZE && c >= -P::W && c < 64 + P::E) return;
    if (bad++ < 20) printf("h%d v%d rows %d: %s at row %d column %d\n", H, V, RW, what, r, c);
}

template <int H, int V, int RW>
void walk()
{
    using S = StagePlanes<H, V, RW>;
    using T = LimitPlanes<H, V, RW>;
    constexpr int HH = S::HH, TJ = S::TJ;
    for (int w = 0; w < NWAVE; w++)
        for (int L = 0; L < 64; L++) {
            const int he = L & 7, hr = (L >> 3) & 1, hcol = he < HH ? he - HH : 64 + he - HH;
            {  // k_std_stage
                using P = typename S::P;
                const int ra = RW * w;
                const bool last = w == NWAVE - 1;
                if (w < 2 * HH) in_plane<P>("stage halo row", H, V, RW, w < HH ? w - HH : TJ + w - HH, L);
                if (L < 8 * RW && he < P::XH) in_plane<P>("stage halo column", H, V, RW, ra + hr, hcol);
                for (int e = 0; e < RW + (last ? 1 : 0); e++)
                    for (int m = -HH; m < HH; m++) {
                        in_plane<P>("stage y face", H, V, RW, ra + e + m, L);
                        if (e < RW) in_plane<P>("stage x face", H, V, RW, ra + e, L + m);
                    }
            }
            {  // k_std_limit
                using P = typename T::P;
                using B = typename T::B;
                const int ra = RW * w - 1;
                if (w >= 1 && w <= 2 * HH - 1)
                    in_plane<P>("limiter halo row", H, V, RW, w <= HH ? -1 - w : TJ - 2 + w - HH, L);
                if (L < 8 * RW && he < P::XH) in_plane<P>("limiter halo column", H, V, RW, ra + hr, hcol);
                if (L < 8 * RW && he >= 6) in_plane<B>("base halo column", H, V, RW, ra + hr, -1);
                if (w >= NWAVE - 2) in_plane<B>("base halo row", H, V, RW, -2, L);
                for (int e = 0; e < RW; e++) {
                    for (int m = -HH; m < HH; m++) {
                        in_plane<P>("limiter y face", H, V, RW, ra + e + m, L);
                        in_plane<P>("limiter x face", H, V, RW, ra + e, L + m);
                    }
                    in_plane<B>("base cell", H, V, RW, ra + e, L);
                    in_plane<B>("base west", H, V, RW, ra + e, L - 1);
                    in_plane<B>("base south", H, V, RW, ra + e - 1, L);
                    in_plane<B>("base north", H, V, RW, ra + e + 1, L);
                }
            }
        }
}

template <int H>
void orders()
{
    walk<H, 1, 1>(), walk<H, 1, 2>();
    walk<H, 3, 1>(), walk<H, 3, 2>();
    walk<H, 5, 1>(), walk<H, 5, 2>();
}

int main()
{
    orders<1>(), orders<3>(), orders<5>();
    printf("%d accesses outside their plane\n", bad);
    return bad != 0;
}
