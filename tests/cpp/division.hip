// div_by against the machine's division: every divisor up to 4096 and around powers of two, at
// and beside multiples of it up to 2^31 - 1
#include "lt_device.hpp"

#include <cstdio>

int main()
{
    const long long top = 2147483647ll;
    auto check = [&](long long d) {
        const lt::Div v = lt::make_div((int)d);
        for (long long k = 0; k < 200; ++k)
            for (long long q : {k, top / d - k, (top / d) * k / 200})
                for (long long n = q * d - 1; n <= q * d + 1; ++n) {
                    if (n < 0 || n > top) continue;
                    int r = (int)n;
                    if (lt::div_by((int)n, v) != n / d || lt::mod_div(r, v) != n % d || r != n / d) {
                        std::printf("%lld / %lld\n", n, d);
                        return false;
                    }
                }
        return true;
    };
    for (long long d = 1; d <= 4096; ++d)
        if (!check(d)) return 1;
    for (int b = 12; b < 31; ++b)
        for (long long d = (1ll << b) - 2; d <= (1ll << b) + 2; ++d)
            if (!check(d)) return 1;
    return check(top) ? 0 : 1;
}
