// finish_threads for the triples (pairs, pairs with a group of 192 atoms or more,
// largest group) of the command line.
#include <stdio.h>
#include <stdlib.h>

#include "fo_internal.h"

int main(int argc, char** argv) {
  for (int i = 1; i + 2 < argc; i += 3)
    printf("%d ", fo::finish_threads(atoi(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2])));
}
