// Takes and gives room on a GPU's account as one process of its own, by lines on
// stdin: "take N" (answers 1 or 0), "give N" (answers 1); ends with the input.
// Its first line of output says that the account is open.
#include "../wavi.jl_amd/csrc/wavi_room.h"

#include <cstdio>
#include <cstdlib>

int main(int argc, char **argv)
{
    if (argc != 3) return 2;
    wavi::Room room;
    room.open(argv[1], atoi(argv[2]));
    puts("open");
    fflush(stdout);
    char verb[16];
    int n;
    while (scanf("%15s %d", verb, &n) == 2) {
        bool ok = true;
        if (verb[0] == 't')
            ok = room.take(n);
        else
            room.give(n);
        printf("%d\n", ok ? 1 : 0);
        fflush(stdout);
    }
    return 0;
}
