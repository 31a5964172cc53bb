// Answers of the library's dispatch rules, one line per line of standard input:
//   visc TILES KTOT FP64 LIMITS SURFACE MASON   levels per block of the viscosity kernel
//   row N ROWS                                  lanes per row, values per lane and butterflies of a
//                                               launch over ROWS rows of N points, or "none"
//   batch SIZE                                  bytes of an argument buffer made for SIZE bytes
#include <iostream>
#include <sstream>

#include "mhh_batch.h"
#include "mhh_rowfft.h"

int main()
{
    std::string line, what;
    while (std::getline(std::cin, line))
    {
        std::istringstream in(line);
        in >> what;
        if (what == "visc")
        {
            int tiles, ktot, fp64, limits, sfc, mason;
            in >> tiles >> ktot >> fp64 >> limits >> sfc >> mason;
            std::cout << mhh::march_kchunk(tiles, ktot, mhh::MARCH_LEAST_VISC, mhh::visc_most(fp64, limits, sfc, mason));
        }
        else if (what == "row")
        {
            int n;
            long long rows;
            mhh::Row_plan p;
            in >> n >> rows;
            if (!mhh::make_row_plan(n, rows, p)) std::cout << "none";
            else std::cout << (1 << p.lsh) << " " << p.vals << " " << (p.arith == mhh::ROW_DIRECT ? "direct" : "radix8");
        }
        else if (what == "batch")
        {
            size_t size;
            in >> size;
            std::cout << mhh::batch_capacity(size);
        }
        std::cout << "\n";
    }
}
