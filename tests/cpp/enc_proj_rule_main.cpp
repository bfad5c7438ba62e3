// Host-only driver of csrc/enc_proj_rule.h: reads "rows J n_cu" lines, prints the kernel each takes.
#include <cstdio>

#include "enc_proj_rule.h"

int main() {
    long long rows;
    int J, n_cu;
    while (scanf("%lld %d %d", &rows, &J, &n_cu) == 3) printf("%c\n", pkhost::enc_proj_kernel_for(rows, J, n_cu));
    return 0;
}
